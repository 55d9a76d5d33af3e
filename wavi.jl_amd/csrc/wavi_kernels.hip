// wavi_kernels.hip - gfx950 kernels of the WAVI.jl velocity solve.
//
// Layout: every field is a full grid in HBM, x fastest (u: (nx+1) x ny,
// v: nx x (ny+1), h: nx x ny, c: (nx-1) x (ny-1), sigma: nx x ny x nsigma
// with sigma slowest).  Vectors of the reference's "inner" unknowns are full
// u/v grids that are zero off the inner masks, so no gather/scatter index
// maps exist on the device.
//
// Kernels named k_tile_* run one 256-thread workgroup per 16 x 16 block of
// the u grid and of the v grid (grid (nbx, nby)); they own the Haar blocks
// (levels <= 3) and write one reduction partial per block.  Other kernels
// are flat (256 threads, one point each).
#include <type_traits>
#include "wavi_device.h"

namespace wavi {

// ===========================================================================
// small utilities

// p[k] where ok, else dflt, with the load issued unconditionally (at index 0
// where !ok; every array here holds at least one element, the grid being at
// least 2 x 2): a guarded load becomes a branch with a wait of its own, so
// that a launch's loads would go out one round trip after another.
template <typename V>
__device__ __forceinline__ V ld_or(bool ok, const V *p, int k, V dflt)
{
    const V v = p[ok ? k : 0];
    return ok ? v : dflt;
}

template <typename T>
__global__ void k_fill(T *a, T v, int n)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) a[k] = v;
}

// u / v pairs of the elementwise kernels above in one launch: blockIdx.y
// selects the u (0) or v (1) arrays.
template <typename Tin, typename Tout>
__global__ void k_select_uv(const Tin *iu, const uint8_t *mu, Tout *ou, int nu, const Tin *iv, const uint8_t *mv,
                            Tout *ov, int nv)
{
    const bool v = blockIdx.y != 0;
    const Tin *in = v ? iv : iu;
    const uint8_t *mask = v ? mv : mu;
    Tout *out = v ? ov : ou;
    const int n = v ? nv : nu;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) out[k] = mask[k] ? (Tout)in[k] : Tout(0);
}

template <typename T>
__global__ void k_copy_masked_uv(T *du, const T *su, const uint8_t *mu, int nu, T *dv, const T *sv,
                                 const uint8_t *mv, int nv)
{
    const bool v = blockIdx.y != 0;
    T *dst = v ? dv : du;
    const T *src = v ? sv : su;
    const uint8_t *mask = v ? mv : mu;
    const int n = v ? nv : nu;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n && mask[k]) dst[k] = src[k];
}

__global__ void k_set_velocities_uv(double *U, const double *xu, const double *eu, const uint8_t *iu, int nu,
                                    double *V, const double *xv, const double *ev, const uint8_t *iv, int nv)
{
    const bool v = blockIdx.y != 0;
    double *W = v ? V : U;
    const double *x = v ? xv : xu, *e = v ? ev : eu;
    const uint8_t *inner = v ? iv : iu;
    const int n = v ? nv : nu;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n && inner[k]) W[k] = x[k] + e[k];
}

template <typename T>
__global__ void k_fill_uv(T *au, int nu, T *av, int nv, T val)
{
    const bool v = blockIdx.y != 0;
    T *a = v ? av : au;
    const int n = v ? nv : nu;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) a[k] = val;
}

// Up to CONV_MAX conversions in one launch: blockIdx.y selects the array.
constexpr int CONV_MAX = 12;
template <typename Tin, typename Tout>
struct ConvList {
    const Tin *in[CONV_MAX];
    Tout *out[CONV_MAX];
    int n[CONV_MAX];
};

template <typename Tin, typename Tout>
__global__ void k_convert_list(ConvList<Tin, Tout> L)
{
    const int a = blockIdx.y;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < L.n[a]) L.out[a][k] = (Tout)L.in[a][k];
}

// out = mask ? in : 0
template <typename Tin, typename Tout>
__global__ void k_select(const Tin *in, const uint8_t *mask, Tout *out, int n)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) out[k] = mask[k] ? (Tout)in[k] : Tout(0);
}

// dst = src where mask
template <typename T>
__global__ void k_copy_masked(T *dst, const T *src, const uint8_t *mask, int n)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n && mask[k]) dst[k] = src[k];
}

// mask as 0.0/1.0 <-> uint8
__global__ void k_mask_from_double(const double *m, uint8_t *out, int n)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) out[k] = m[k] > 0.5 ? 1 : 0;
}

__global__ void k_mask_to_double(const uint8_t *m, double *out, int n)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) out[k] = m[k] ? 1.0 : 0.0;
}

// ===========================================================================
// Canonical [u; v] dot-product partials: one per 16x16 block (u blocks then
// v blocks).  b == nullptr gives sum of squares.
template <typename T>
__global__ void k_tile_dot(GridDims g, const T *au, const T *av, const T *bu, const T *bv, double *P)
{
    __shared__ double lds[256];
    const int lx = threadIdx.x & 15, ly = threadIdx.x >> 4;
    const int bx = blockIdx.x, by = blockIdx.y;
    const int i = bx * TILE + lx, j = by * TILE + ly;
    if (bx < g.nbxu && by < g.nbyu) {
        double v = 0.0;
        if (i < g.nxu && j < g.nyu) {
            int k = i + g.nxu * j;
            v = bu ? (double)au[k] * (double)bu[k] : (double)au[k] * (double)au[k];
        }
        double s = tree256(v, lds);
        if (threadIdx.x == 0) P[bx + g.nbxu * by] = s;
    }
    if (bx < g.nbxv && by < g.nbyv) {
        double v = 0.0;
        if (i < g.nxv && j < g.nyv) {
            int k = i + g.nxv * j;
            v = bv ? (double)av[k] * (double)bv[k] : (double)av[k] * (double)av[k];
        }
        double s = tree256(v, lds);
        if (threadIdx.x == 0) P[g.nbxu * g.nbyu + bx + g.nbxv * by] = s;
    }
}

// out[slot] = sqrt(sum of partials) for each of `count` partial arrays.
__global__ void k_finish_norms(const double *P0, const double *P1, int np, double *out)
{
    __shared__ double lds[256];
    double a = lanes_sum(P0, np, lds);
    double b = P1 ? lanes_sum(P1, np, lds) : 0.0;
    if (threadIdx.x == 0) {
        out[0] = sqrt(a);
        out[1] = sqrt(b);
    }
}

// out[c] = sum of partial array c (P + c * np), c < count (no square root)
__global__ void k_finish_sums(const double *P, int np, int count, double *out)
{
    __shared__ double lds[256];
    for (int c = 0; c < count; ++c) {
        double a = lanes_sum(P + (size_t)c * np, np, lds);
        if (threadIdx.x == 0) out[c] = a;
        __syncthreads();
    }
}

// flexible CG: x += alpha p, r -= alpha q on the u then the v grid
__global__ void k_fcg_step(int nu, int nv, double alpha, double *xu, double *xv, double *ru, double *rv,
                           const double *pu, const double *pv, const double *qu, const double *qv)
{
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < nu) {
        xu[t] = xu[t] + alpha * pu[t];
        ru[t] = ru[t] - alpha * qu[t];
    } else if (t < nu + nv) {
        t -= nu;
        xv[t] = xv[t] + alpha * pv[t];
        rv[t] = rv[t] - alpha * qv[t];
    }
}

// flexible CG: p = z + beta p at inner points, 0 elsewhere
__global__ void k_fcg_dir(int nu, int nv, double beta, const uint8_t *ui, const uint8_t *vi, const double *zu,
                          const double *zv, double *pu, double *pv)
{
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < nu) {
        pu[t] = ui[t] ? zu[t] + beta * pu[t] : 0.0;
    } else if (t < nu + nv) {
        t -= nu;
        pv[t] = vi[t] ? zv[t] + beta * pv[t] : 0.0;
    }
}

// ===========================================================================
// update_state! steps before the solve (src/Models/update_state.jl:51-147).

struct GeomArgs {
    const uint8_t *hm, *um, *vm;
    const double *b, *h;
    double *s, *haf, *q;  // q: 4 quadrant fractions, 4*nh
    double *gfh, *gfu, *gfv;
    double *hu, *su, *hv, *sv;
    double *wc, *dsdh, *acc, *mel;
    const double *wc_param, *acc_param;
    double sl, ri, rw, melt;
};

// update_surface_elevation! (:51-57), update_height_above_floatation! (:80-85)
__global__ void k_surface_haf(GridDims g, GeomArgs a)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= g.nx * g.ny) return;
    double h = a.h[k], b = a.b[k];
    if (a.hm[k]) {
        double s1 = b + h, s2 = a.sl + h * (1.0 - a.ri / a.rw);
        double s = s1 > s2 ? s1 : s2;
        if (__builtin_isnan(s1) || __builtin_isnan(s2)) s = __builtin_nan("");
        a.s[k] = s;
    }
    a.haf[k] = h - (a.rw / a.ri) * (a.sl - b);
}

// pos_fraction quadrant area (src/utilities.jl:263-360) of one cell from the
// values at the cell (v1, its mask m1) and at the quadrant's two neighbours
// (z2, z3 with masks m2, m3; an unmasked neighbour takes the cell's value).
__device__ __forceinline__ double pos_fraction_area(double v1, bool m1, double z2, bool m2, double z3, bool m3)
{
    double v2 = m2 ? z2 : v1;
    double v3 = m3 ? z3 : v1;
    double s1 = (v1 > 0) - (v1 < 0), s2 = (v2 > 0) - (v2 < 0), s3 = (v3 > 0) - (v3 < 0);
    double area = 0.0;
    if (!((s1 == s2) && (s1 == s3))) {
        bool flip = fabs(v3 - v1) < fabs(v2 - v1);
        double a, b;
        if (!flip) {
            a = -(v2 - v1) / (v3 - v1);
            b = -2.0 * v1 / (v3 - v1);
        } else {
            a = -(v3 - v1) / (v2 - v1);
            b = -2.0 * v1 / (v2 - v1);
        }
        double a1 = 0.5 * (b * b) / a;
        double a2 = 0.5 * ((1.0 - b) * (1.0 - b)) / a;
        double a3 = 0.5 * a + b;
        int t1 = (b > 0.0) + (b > 1.0);
        double ab = a + b;
        int t2 = (ab > 0.0) + (ab > 1.0);
        int ix = 1 + t1 + 3 * t2;
        switch (ix) {
        case 1: area = 0.0; break;
        case 2: area = -a1; break;
        case 3: area = a2 - a1; break;
        case 4: area = a1 + a3; break;
        case 5: area = a3; break;
        case 6: area = a2 + a3; break;
        case 7: area = (1.0 - a2) + a1; break;
        case 8: area = 1.0 - a2; break;
        default: area = 1.0; break;
        }
        if (b < 0.0) area = 1.0 - area;
        if (v1 < 0.0) area = 1.0 - area;
    }
    if (v1 > 0.0 && v2 > 0.0 && v3 > 0.0) area = 1.0;
    if (v1 <= 0.0 && v2 <= 0.0 && v3 <= 0.0) area = 0.0;
    if (!m1) area = 0.0;
    return area;
}


// update_grounded_fraction (:92-99) on h, then accumulation, melt,
// weertman_c and dsdh (:106-147)
__global__ void k_gf_h(GridDims g, GeomArgs a)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    const int nh = g.nx * g.ny;
    if (k >= nh) return;
    int i = k % g.nx, j = k / g.nx;
    // the cell and its four neighbours (clamped), every load before the
    // first store
    const int M = g.nx, N = g.ny;
    const int kE = (i + 1 < M ? i + 1 : M - 1) + M * j, kW = (i > 0 ? i - 1 : 0) + M * j;
    const int kN = i + M * (j + 1 < N ? j + 1 : N - 1), kS = i + M * (j > 0 ? j - 1 : 0);
    const double zc = a.haf[k], zE = a.haf[kE], zN = a.haf[kN], zW = a.haf[kW], zS = a.haf[kS];
    const bool mc = a.hm[k], mE = a.hm[kE], mN = a.hm[kN], mW = a.hm[kW], mS = a.hm[kS];
    const double accp = a.acc_param[k], wcp = a.wc_param[k];
    // quadrants 1..4 take points (2, 3) = (E, N), (N, W), (W, S), (S, E),
    // each clamped to the cell at the grid's edge (utilities.jl:263-360)
    const double q[4] = {pos_fraction_area(zc, mc, zE, mE, zN, mN), pos_fraction_area(zc, mc, zN, mN, zW, mW),
                         pos_fraction_area(zc, mc, zW, mW, zS, mS), pos_fraction_area(zc, mc, zS, mS, zE, mE)};
    double af = 0.0;
#pragma unroll
    for (int quad = 1; quad <= 4; ++quad) {
        a.q[(quad - 1) * nh + k] = q[quad - 1];
        af = af + 0.25 * q[quad - 1];
    }
    a.gfh[k] = af;
    a.acc[k] = accp;
    a.mel[k] = a.melt;
    a.wc[k] = wcp * af;
    a.dsdh[k] = (1.0 - a.ri / a.rw) + (a.ri / a.rw) * af;
}

// masked h -> face averages of update_geometry_on_uv_grids! (:65-73) and the
// u/v grounded fractions of pos_fraction (utilities.jl:367-390)
__global__ void k_geom_uv(GridDims g, GeomArgs a)
{
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int nu = g.nxu * g.nyu, nv = g.nxv * g.nyv, nh = g.nx * g.ny;
    const int nx = g.nx, ny = g.ny;
    if (t >= nu + nv) return;
    // the face between h cells ka (left / below) and kb; every load issued
    // before the first is used (ld_or), the sums in the same order as before
    const bool v = t >= nu;
    const int tt = v ? t - nu : t;
    const int i = v ? tt % g.nxv : tt % g.nxu, j = v ? tt / g.nxv : tt / g.nxu;
    const bool oka = v ? j >= 1 : i >= 1, okb = v ? j < ny : i < nx;
    const int ka = v ? i + nx * (j - 1) : (i - 1) + nx * j, kb = i + nx * j;
    // grounded fraction: on u quadrants 1, 4 from cell i - 1 and 2, 3 from
    // cell i; on v quadrants 1, 2 from cell j - 1 and 3, 4 from cell j
    const double q1 = ld_or(oka, a.q, ka, 0.0);
    const double q2 = v ? ld_or(oka, a.q, nh + ka, 0.0) : ld_or(okb, a.q, nh + kb, 0.0);
    const double q3 = ld_or(okb, a.q, 2 * nh + kb, 0.0);
    const double q4 = v ? ld_or(okb, a.q, 3 * nh + kb, 0.0) : ld_or(oka, a.q, 3 * nh + ka, 0.0);
    const bool fm = (v ? a.vm : a.um)[tt];
    const uint8_t ha = ld_or(oka, a.hm, ka, (uint8_t)0), hb = ld_or(okb, a.hm, kb, (uint8_t)0);
    const double hha = ld_or(oka, a.h, ka, 0.0), hhb = ld_or(okb, a.h, kb, 0.0);
    const double sa = ld_or(oka, a.s, ka, 0.0), sb = ld_or(okb, a.s, kb, 0.0);
    double gf = 0.0;
    gf = gf + 0.25 * q1;
    gf = gf + 0.25 * q2;
    gf = gf + 0.25 * q3;
    gf = gf + 0.25 * q4;
    (v ? a.gfv : a.gfu)[tt] = gf;
    if (fm) {
        double den = 0.0, nh_ = 0.0, ns_ = 0.0;
        if (oka) {
            den = den + 0.5 * (double)ha;
            nh_ = nh_ + 0.5 * (ha ? hha : 0.0);
            ns_ = ns_ + 0.5 * (ha ? sa : 0.0);
        }
        if (okb) {
            den = den + 0.5 * (double)hb;
            nh_ = nh_ + 0.5 * (hb ? hhb : 0.0);
            ns_ = ns_ + 0.5 * (hb ? sb : 0.0);
        }
        (v ? a.hv : a.hu)[tt] = nh_ / den;
        (v ? a.sv : a.su)[tt] = ns_ / den;
    }
}

// ===========================================================================
// inner_update! (src/Models/update_velocities.jl:32-45, 202-383)

struct InnerArgs {
    const uint8_t *hm, *um, *vm, *cm;
    const double *U, *V;
    const double *h, *wc, *gfh, *gfu, *gfv, *dsdh, *glen_b;
    const double *zeta, *qw;       // nsigma
    double *sr, *avs, *bs, *beta, *tau, *eta, *etaav, *f1, *f2, *beff;
    double *bu, *bv;
    double *heta_h, *heta_c, *dimp;
    double rdx, rdy;
    double wexp, wreg2, gexp, greg2, c0;
    int ns, niter_visc, xfirst_c2h, yfirst_h2c;
};

// shear strain (uy + vx) on the c mask at corner (a, b), 0 outside the c grid
__device__ __forceinline__ double corner_shear(const GridDims &g, const InnerArgs &p, int a, int b)
{
    const int nxc = g.nx - 1, nyc = g.ny - 1;
    const bool in = a >= 0 && a < nxc && b >= 0 && b < nyc;
    const int nxu = g.nxu, nx = g.nx;
    // every load issued at once (ld_or), values selected
    const int ku1 = (a + 1) + nxu * (b + 1), ku0 = (a + 1) + nxu * b;
    const int kv1 = (a + 1) + nx * (b + 1), kv0 = a + nx * (b + 1);
    const bool cm = ld_or(in, p.cm, a + nxc * b, (uint8_t)0) != 0;
    const bool mu1 = ld_or(in, p.um, ku1, (uint8_t)0) != 0, mu0 = ld_or(in, p.um, ku0, (uint8_t)0) != 0;
    const bool mv1 = ld_or(in, p.vm, kv1, (uint8_t)0) != 0, mv0 = ld_or(in, p.vm, kv0, (uint8_t)0) != 0;
    const double U1 = ld_or(in, p.U, ku1, 0.0), U0 = ld_or(in, p.U, ku0, 0.0);
    const double V1 = ld_or(in, p.V, kv1, 0.0), V0 = ld_or(in, p.V, kv0, 0.0);
    const double u1 = mu1 ? U1 : 0.0, u0 = mu0 ? U0 : 0.0;
    const double v1 = mv1 ? V1 : 0.0, v0 = mv0 ? V0 : 0.0;
    const double dudy = p.rdy * u1 - p.rdy * u0;
    const double dvdx = p.rdx * v1 - p.rdx * v0;
    return (in && cm) ? dudy + dvdx : 0.0;
}

// gc.cent (CGrid.jl:45) at h cell (i, j) in the reference's factor order
__device__ __forceinline__ double cent_c_to_h(const GridDims &g, const InnerArgs &p, int i, int j)
{
    const int nxc = g.nx - 1, nyc = g.ny - 1;
    // the four corners' loads first, then the sums in the reference's order
    const double s00 = corner_shear(g, p, i - 1, j - 1), s10 = corner_shear(g, p, i, j - 1);
    const double s01 = corner_shear(g, p, i - 1, j), s11 = corner_shear(g, p, i, j);
    double out = 0.0;
    if (p.xfirst_c2h) {
        if (j - 1 >= 0 && j - 1 < nyc) {
            double t0 = 0.0;
            if (i - 1 >= 0 && i - 1 < nxc) t0 = t0 + 0.5 * s00;
            if (i >= 0 && i < nxc) t0 = t0 + 0.5 * s10;
            out = out + 0.5 * t0;
        }
        if (j >= 0 && j < nyc) {
            double t1 = 0.0;
            if (i - 1 >= 0 && i - 1 < nxc) t1 = t1 + 0.5 * s01;
            if (i >= 0 && i < nxc) t1 = t1 + 0.5 * s11;
            out = out + 0.5 * t1;
        }
    } else {
        if (i - 1 >= 0 && i - 1 < nxc) {
            double t0 = 0.0;
            if (j - 1 >= 0 && j - 1 < nyc) t0 = t0 + 0.5 * s00;
            if (j >= 0 && j < nyc) t0 = t0 + 0.5 * s01;
            out = out + 0.5 * t0;
        }
        if (i >= 0 && i < nxc) {
            double t1 = 0.0;
            if (j - 1 >= 0 && j - 1 < nyc) t1 = t1 + 0.5 * s10;
            if (j >= 0 && j < nyc) t1 = t1 + 0.5 * s11;
            out = out + 0.5 * t1;
        }
    }
    return out;
}

// All h-cell updates of inner_update!: strain rate, speeds, beta, basal drag,
// viscosity on the sigma levels, quadratures, beta_eff and the h-grid
// rheological coefficients.
constexpr int INNER_NS_PREFETCH = 8;  // sigma levels whose eta and glen_b k_inner_h loads up front

__global__ void k_inner_h(GridDims g, InnerArgs p)
{
    const int nh = g.nx * g.ny;
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nh) return;
    const int i = k % g.nx, j = k / g.nx;
    const int nxu = g.nxu, nx = g.nx;
    // every load of the cell issued before the first is used: masks with
    // their fields (the values selected), the shear's corners, and eta and
    // glen_b on up to INNER_NS_PREFETCH levels
    const bool hm = p.hm[k];
    const double Ua = p.U[i + nxu * j], Ub = p.U[(i + 1) + nxu * j];
    const double Va = p.V[i + nx * j], Vb = p.V[i + nx * (j + 1)];
    const bool ma = p.um[i + nxu * j], mb = p.um[(i + 1) + nxu * j];
    const bool na = p.vm[i + nx * j], nb = p.vm[i + nx * (j + 1)];
    const double shc = cent_c_to_h(g, p, i, j);
    double eta_k[INNER_NS_PREFETCH], gb_k[INNER_NS_PREFETCH], zeta_k[INNER_NS_PREFETCH], qw_k[INNER_NS_PREFETCH];
#pragma unroll
    for (int ks = 0; ks < INNER_NS_PREFETCH; ++ks) {
        eta_k[ks] = ld_or(ks < p.ns, p.eta, k + nh * ks, 0.0);
        gb_k[ks] = ld_or(ks < p.ns, p.glen_b, k + nh * ks, 0.0);
        zeta_k[ks] = ld_or(ks < p.ns, p.zeta, ks, 0.0);
        qw_k[ks] = ld_or(ks < p.ns, p.qw, ks, 0.0);
    }
    // (and before the first store, which the compiler cannot move them past)
    const double f2_old = p.f2[k], beta_old = p.beta[k], wck = p.wc[k], hk = p.h[k], dsdhk = p.dsdh[k];
    // update_shelf_strain_rate! (:202-209)
    double ux = 0.0, vy = 0.0, sh = 0.0;
    double ub = 0.0, vb = 0.0;
    {
        double u0 = ma ? Ua : 0.0;
        double u1 = mb ? Ub : 0.0;
        double v0 = na ? Va : 0.0;
        double v1 = nb ? Vb : 0.0;
        if (hm) {
            ux = p.rdx * u1 - p.rdx * u0;
            vy = p.rdy * v1 - p.rdy * v0;
            sh = shc;
            ub = 0.5 * u0 + 0.5 * u1;
            vb = 0.5 * v0 + 0.5 * v1;
        }
    }
    double sr = sqrt(((ux * ux + vy * vy) + ux * vy) + 0.25 * (sh * sh));
    p.sr[k] = sr;
    // update_av_speed! (:216-220)
    double avs = sqrt(ub * ub + vb * vb);
    p.avs[k] = avs;
    // update_bed_speed!, update_β!, update_basal_drag! (:227-255)
    double bs = avs / (1.0 + f2_old * beta_old);
    double beta = wck * det_pow(sqrt(bs * bs + p.wreg2), p.wexp);
    double tau = beta * bs;
    p.bs[k] = bs;
    p.beta[k] = beta;
    p.tau[k] = tau;
    // inner_update_viscosity!, update_av_viscosity!, update_quadrature_falpha! (:264-328)
    double av = 0.0, q1 = 0.0, q2 = 0.0;
    if (hm) {
        // level ks from its eta, glen_b, zeta and weight (the levels in
        // increasing order: the prefetched ones unrolled, then any others)
        auto level = [&](int ks, double eta, double gb, double zeta, double w) {
            for (int it = 0; it < p.niter_visc; ++it) {
                double q = (tau * zeta) / eta;
                double arg = sqrt((sr * sr + 0.25 * (q * q)) + p.greg2);
                eta = (0.5 * gb) * det_pow(arg, p.gexp);
            }
            p.eta[k + nh * ks] = eta;
            av = av + w * eta;
            q1 = q1 + ((w * hk) * zeta) / eta;
            q2 = q2 + ((w * hk) * (zeta * zeta)) / eta;
        };
#pragma unroll
        for (int ks = 0; ks < INNER_NS_PREFETCH; ++ks)
            if (ks < p.ns) level(ks, eta_k[ks], gb_k[ks], zeta_k[ks], qw_k[ks]);
        for (int ks = INNER_NS_PREFETCH; ks < p.ns; ++ks)
            level(ks, p.eta[k + nh * ks], p.glen_b[k + nh * ks], p.zeta[ks], p.qw[ks]);
    }
    p.etaav[k] = av;
    p.f1[k] = q1;
    p.f2[k] = q2;
    // update_βeff! (:335-339)
    p.beff[k] = beta / (1.0 + q2 * beta);
    // update_rheological_operators! (:374-383), h-grid parts
    p.heta_h[k] = hm ? hk * av : 0.0;
    p.dimp[k] = hm ? p.c0 * dsdhk : 0.0;
}

// update_βeff_on_uv_grids! (:348-366) and the c-grid coefficient
// gc.dneghηav (:378)
__global__ void k_inner_uvc(GridDims g, InnerArgs p)
{
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int nu = g.nxu * g.nyu, nv = g.nxv * g.nyv, nc = (g.nx - 1) * (g.ny - 1);
    const int nx = g.nx;
    if (t < nu + nv) {
        // the face between h cells ka (left / below) and kb; every load
        // issued before the first is used (ld_or), the sums as before
        const bool v = t >= nu;
        const int tt = v ? t - nu : t;
        const int i = v ? tt % g.nxv : tt % g.nxu, j = v ? tt / g.nxv : tt / g.nxu;
        const bool oka = v ? j >= 1 : i >= 1, okb = v ? j <= g.ny - 1 : i <= nx - 1;
        const int ka = v ? i + nx * (j - 1) : (i - 1) + nx * j, kb = i + nx * j;
        const bool fm = (v ? p.vm : p.um)[tt];
        const double gff = (v ? p.gfv : p.gfu)[tt];
        const uint8_t ha = ld_or(oka, p.hm, ka, (uint8_t)0), hb = ld_or(okb, p.hm, kb, (uint8_t)0);
        const double ba = ld_or(oka, p.beff, ka, 0.0), bb = ld_or(okb, p.beff, kb, 0.0);
        const double ga = ld_or(oka, p.gfh, ka, 0.0), gb = ld_or(okb, p.gfh, kb, 0.0);
        if (!fm) return;
        double den = 0.0, nb = 0.0, ng = 0.0;
        if (oka) {
            den = den + 0.5 * (double)ha;
            nb = nb + 0.5 * (ha ? ba : 0.0);
            ng = ng + 0.5 * (ha ? ga : 0.0);
        }
        if (okb) {
            den = den + 0.5 * (double)hb;
            nb = nb + 0.5 * (hb ? bb : 0.0);
            ng = ng + 0.5 * (hb ? gb : 0.0);
        }
        double b = nb / den;
        double ip = ng / den;
        if (ip > 0.0) b = (b * gff) / ip;
        (v ? p.bv : p.bu)[tt] = b;
    } else if (t < nu + nv + nc) {
        int tc = t - nu - nv;
        int i = tc % (nx - 1), j = tc / (nx - 1);
        // the four cells' h and eta_av loaded with the corner's mask
        const int k00 = i + nx * j, k10 = k00 + 1, k01 = k00 + nx, k11 = k01 + 1;
        const double h00 = p.h[k00], h10 = p.h[k10], h01 = p.h[k01], h11 = p.h[k11];
        const double e00 = p.etaav[k00], e10 = p.etaav[k10], e01 = p.etaav[k01], e11 = p.etaav[k11];
        if (!p.cm[tc]) {
            p.heta_c[tc] = 0.0;
            return;
        }
        // gh.cent_xy (HGrid.jl:203) of h*eta_av in the reference's factor order
        double a00 = h00 * e00;
        double a10 = h10 * e10;
        double a01 = h01 * e01;
        double a11 = h11 * e11;
        double out;
        if (p.yfirst_h2c) {
            double t0 = 0.5 * a00 + 0.5 * a01;
            double t1 = 0.5 * a10 + 0.5 * a11;
            out = 0.5 * t0 + 0.5 * t1;
        } else {
            double t0 = 0.5 * a00 + 0.5 * a10;
            double t1 = 0.5 * a01 + 0.5 * a11;
            out = 0.5 * t0 + 0.5 * t1;
        }
        p.heta_c[tc] = out;
    }
}

// ===========================================================================
// Reverse of one Picard iteration, for the adjoint basal-drag gradient (no
// reference counterpart).  Iteration k is inner_update! from the state
// (u_{k-1}, eta, beta, f2 of checkpoint k-1), then u_k = A_k^{-1} b.  With
// lambda_k = A_k^{-1} ubar_k, the coefficient adjoints are
// cbar = -d(lambda^T A(c) u_k)/dc, and the chain rule runs back through
// update_rheological_operators!, update_βeff_on_uv_grids!, update_βeff!,
// the quadratures, the viscosity passes, update_basal_drag!, update_β!,
// update_bed_speed!, update_av_speed! and update_shelf_strain_rate!
// (update_velocities.jl:202-383).  k_adj_h does the per-cell part, k_adj_uv
// the gathers onto u_{k-1} and v_{k-1}.

struct AdjArgs {
    InnerArgs p;                               // iteration k recomputed; p.U, p.V = u_{k-1}
    const double *uk, *vk;                     // u_k
    const double *lu, *lv;                     // lambda_k
    const double *eta_old, *beta_old, *f2_old; // checkpoint k-1
    double *etab, *betab, *f2b;                // state adjoints: leaving k on entry, entering k on exit
    double *wcb;                               // += dJ/d(weertman_c on h)
    double *cub, *cvb, *uxb, *vyb, *shb;       // per h cell, for k_adj_uv
    double *ubar, *vbar;                       // out: adjoint of u_{k-1} at inner points
};

// (du/dy + dv/dx) of (U, V) at corner (a, b), unmasked as op_fun! reads it
__device__ __forceinline__ double corner_rate(const GridDims &g, const double *U, const double *V, double rdx,
                                              double rdy, int a, int b)
{
    const int nxu = g.nxu, nx = g.nx;
    return (rdy * U[(a + 1) + nxu * (b + 1)] - rdy * U[(a + 1) + nxu * b]) +
           (rdx * V[(a + 1) + nx * (b + 1)] - rdx * V[a + nx * (b + 1)]);
}

__global__ void k_adj_h(GridDims g, AdjArgs a)
{
    const int nh = g.nx * g.ny;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nh) return;
    const InnerArgs &p = a.p;
    const int nx = g.nx, ny = g.ny, nxu = g.nxu, nxc = g.nx - 1, nyc = g.ny - 1;
    const int i = k % nx, j = k / nx;
    const bool hm = p.hm[k];
    const double rdx = p.rdx, rdy = p.rdy;
    // update_rheological_operators!: h eta_av on h, and cent onto c
    double hqb = 0.0;
    if (hm) {
        const double dudx = rdx * a.uk[(i + 1) + nxu * j] - rdx * a.uk[i + nxu * j];
        const double dvdy = rdy * a.vk[i + nx * (j + 1)] - rdy * a.vk[i + nx * j];
        const double dlx = rdx * a.lu[(i + 1) + nxu * j] - rdx * a.lu[i + nxu * j];
        const double dly = rdy * a.lv[i + nx * (j + 1)] - rdy * a.lv[i + nx * j];
        hqb = 2.0 * (2.0 * dudx + dvdy) * dlx + 2.0 * (2.0 * dvdy + dudx) * dly;
    }
    for (int b = j - 1; b <= j; ++b)
        for (int c = i - 1; c <= i; ++c)
            if (c >= 0 && c < nxc && b >= 0 && b < nyc && p.cm[c + nxc * b])
                hqb += 0.25 * (corner_rate(g, a.uk, a.vk, rdx, rdy, c, b) *
                               corner_rate(g, a.lu, a.lv, rdx, rdy, c, b));
    const double etaavb = p.h[k] * hqb;
    // update_βeff_on_uv_grids!
    double beffb = 0.0;
    if (hm) {
        for (int c = i; c <= i + 1; ++c) {
            const int ku = c + nxu * j;
            if (!p.um[ku]) continue;
            double den = 0.0, ng = 0.0;
            if (c >= 1) {
                den = den + 0.5 * (double)p.hm[(c - 1) + nx * j];
                ng = ng + 0.5 * (p.hm[(c - 1) + nx * j] ? p.gfh[(c - 1) + nx * j] : 0.0);
            }
            if (c <= nx - 1) {
                den = den + 0.5 * (double)p.hm[c + nx * j];
                ng = ng + 0.5 * (p.hm[c + nx * j] ? p.gfh[c + nx * j] : 0.0);
            }
            const double ip = ng / den;
            beffb += (a.lu[ku] * a.uk[ku]) * (0.5 / den) * (ip > 0.0 ? p.gfu[ku] / ip : 1.0);
        }
        for (int b = j; b <= j + 1; ++b) {
            const int kv = i + nx * b;
            if (!p.vm[kv]) continue;
            double den = 0.0, ng = 0.0;
            if (b >= 1) {
                den = den + 0.5 * (double)p.hm[i + nx * (b - 1)];
                ng = ng + 0.5 * (p.hm[i + nx * (b - 1)] ? p.gfh[i + nx * (b - 1)] : 0.0);
            }
            if (b <= ny - 1) {
                den = den + 0.5 * (double)p.hm[i + nx * b];
                ng = ng + 0.5 * (p.hm[i + nx * b] ? p.gfh[i + nx * b] : 0.0);
            }
            const double ip = ng / den;
            beffb += (a.lv[kv] * a.vk[kv]) * (0.5 / den) * (ip > 0.0 ? p.gfv[kv] / ip : 1.0);
        }
    }
    // update_βeff!: beta_eff = beta / (1 + f2 beta)
    const double beta = p.beta[k], f2 = p.f2[k];
    const double D = 1.0 + f2 * beta;
    double bb = a.betab[k] + beffb / (D * D);
    const double fb = a.f2b[k] - beffb * (beta * beta) / (D * D);
    const double sr = p.sr[k], tau = p.tau[k], bs = p.bs[k];
    double taub = 0.0, srb = 0.0;
    if (hm) {
        for (int s = 0; s < p.ns; ++s) {
            const int k3 = k + nh * s;
            const double z = p.zeta[s], w = p.qw[s], eta = p.eta[k3], gb = p.glen_b[k3];
            // update_av_viscosity!, update_quadrature_falpha!
            double eb = a.etab[k3] + w * etaavb - fb * ((w * p.h[k]) * (z * z)) / (eta * eta);
            // inner_update_viscosity!: the passes from eta_old, then back
            double e[9];
            e[0] = a.eta_old[k3];
            for (int q = 0; q < p.niter_visc; ++q) {
                const double qq = (tau * z) / e[q];
                const double arg = sqrt((sr * sr + 0.25 * (qq * qq)) + p.greg2);
                e[q + 1] = (0.5 * gb) * det_pow(arg, p.gexp);
            }
            for (int q = p.niter_visc - 1; q >= 0; --q) {
                const double qq = (tau * z) / e[q];
                const double arg = sqrt((sr * sr + 0.25 * (qq * qq)) + p.greg2);
                const double gg = eb * e[q + 1] * p.gexp / arg;
                srb += gg * sr / arg;
                const double qb = gg * 0.25 * qq / arg;
                taub += qb * z / e[q];
                eb = -qb * qq / e[q];
            }
            a.etab[k3] = eb;
        }
    }
    // update_basal_drag!: tau = beta bs; update_β!: beta = wc (bs^2 + reg^2)^(wexp/2)
    double bsb = taub * beta;
    bb += taub * bs;
    const double S = bs * bs + p.wreg2;
    a.wcb[k] += bb * det_pow(sqrt(S), p.wexp);
    bsb += bb * beta * p.wexp * bs / S;
    // update_bed_speed!: bs = avs / (1 + f2_old beta_old)
    const double D0 = 1.0 + a.f2_old[k] * a.beta_old[k];
    const double avsb = bsb / D0, avs = p.avs[k];
    a.f2b[k] = -bsb * avs * a.beta_old[k] / (D0 * D0);
    a.betab[k] = -bsb * avs * a.f2_old[k] / (D0 * D0);
    // update_av_speed! and update_shelf_strain_rate! of u_{k-1}
    double cub = 0.0, cvb = 0.0, uxb = 0.0, vyb = 0.0, shb = 0.0;
    if (hm) {
        const double u0 = p.um[i + nxu * j] ? p.U[i + nxu * j] : 0.0;
        const double u1 = p.um[(i + 1) + nxu * j] ? p.U[(i + 1) + nxu * j] : 0.0;
        const double v0 = p.vm[i + nx * j] ? p.V[i + nx * j] : 0.0;
        const double v1 = p.vm[i + nx * (j + 1)] ? p.V[i + nx * (j + 1)] : 0.0;
        if (avs > 0.0) {
            cub = avsb * (0.5 * u0 + 0.5 * u1) / avs;
            cvb = avsb * (0.5 * v0 + 0.5 * v1) / avs;
        }
        if (sr > 0.0) {
            const double ux = rdx * u1 - rdx * u0, vy = rdy * v1 - rdy * v0;
            const double sh = cent_c_to_h(g, p, i, j);
            uxb = srb * (2.0 * ux + vy) / (2.0 * sr);
            vyb = srb * (2.0 * vy + ux) / (2.0 * sr);
            shb = srb * 0.25 * sh / sr;
        }
    }
    a.cub[k] = cub;
    a.cvb[k] = cvb;
    a.uxb[k] = uxb;
    a.vyb[k] = vyb;
    a.shb[k] = shb;
}

// adjoint of the corner shear at c (a, b): cent (c -> h) transposed
__device__ __forceinline__ double adj_corner(const GridDims &g, const AdjArgs &a, int c, int b)
{
    const int nx = g.nx;
    if (!a.p.cm[c + (nx - 1) * b]) return 0.0;
    return 0.25 * (a.shb[c + nx * b] + a.shb[(c + 1) + nx * b] + a.shb[c + nx * (b + 1)] +
                   a.shb[(c + 1) + nx * (b + 1)]);
}

__global__ void k_adj_uv(GridDims g, AdjArgs a)
{
    const int nu = g.nxu * g.nyu, nv = g.nxv * g.nyv;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int nx = g.nx, ny = g.ny;
    const double rdx = a.p.rdx, rdy = a.p.rdy;
    if (t < nu) {
        const int i = t % g.nxu, j = t / g.nxu;
        double s = 0.0;
        if (a.p.um[t]) {
            if (i >= 1) s += 0.5 * a.cub[(i - 1) + nx * j] + rdx * a.uxb[(i - 1) + nx * j];
            if (i <= nx - 1) s += 0.5 * a.cub[i + nx * j] - rdx * a.uxb[i + nx * j];
            if (i >= 1 && i <= nx - 1) {
                if (j >= 1) s += rdy * adj_corner(g, a, i - 1, j - 1);
                if (j <= ny - 2) s -= rdy * adj_corner(g, a, i - 1, j);
            }
        }
        a.ubar[t] = s;
    } else if (t < nu + nv) {
        const int tv = t - nu;
        const int i = tv % g.nxv, j = tv / g.nxv;
        double s = 0.0;
        if (a.p.vm[tv]) {
            if (j >= 1) s += 0.5 * a.cvb[i + nx * (j - 1)] + rdy * a.vyb[i + nx * (j - 1)];
            if (j <= ny - 1) s += 0.5 * a.cvb[i + nx * j] - rdy * a.vyb[i + nx * j];
            if (j >= 1 && j <= ny - 1) {
                if (i >= 1) s += rdx * adj_corner(g, a, i - 1, j - 1);
                if (i <= nx - 2) s -= rdx * adj_corner(g, a, i, j - 1);
            }
        }
        a.vbar[tv] = s;
    }
}

// grad = wc * wcb (dJ/d log C through weertman_c = C * grounded fraction)
__global__ void k_adj_grad(int nh, const double *wc, const double *wcb, double *grad)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < nh) grad[k] = wc[k] * wcb[k];
}

// ===========================================================================
// get_rhs (update_velocities.jl:106-182): f1 + f2 + f3 with f3 = -A(u_fixed)
// passed in as the operator applied to the fixed values.
struct RhsArgs {
    const uint8_t *hm, *ui, *vi;
    const double *s, *dsdh, *acc, *mel;
    const double *hu, *su, *hv, *sv;
    const double *f3u, *f3v;   // A applied to the fixed velocities
    double *bu, *bv;
    double rdx, rdy, g, ri, rw, sl, tdt;
};

__global__ void k_rhs(GridDims g, RhsArgs a)
{
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int nu = g.nxu * g.nyu, nv = g.nxv * g.nyv;
    const int nx = g.nx, ny = g.ny;
    const double rg = a.ri * a.g, hri = 0.5 * a.ri, hrw = 0.5 * a.rw;
    if (t >= nu + nv) return;
    // a face between h cells ka (left / below) and kb: every load issued
    // before the first is used (ld_or), then the reference's f1, f2, f3 terms
    const bool v = t >= nu;
    const int tt = v ? t - nu : t;
    const int i = v ? tt % g.nxv : tt % g.nxu, j = v ? tt / g.nxv : tt / g.nxu;
    const bool oka = v ? j > 0 : i > 0, okb = v ? j < ny : i < nx;
    const int ka = v ? i + nx * (j - 1) : (i - 1) + nx * j, kb = i + nx * j;
    const bool inner = (v ? a.vi : a.ui)[tt];
    const uint8_t ha = ld_or(oka, a.hm, ka, (uint8_t)0), hb = ld_or(okb, a.hm, kb, (uint8_t)0);
    const double sa = ld_or(oka, a.s, ka, 0.0), sb = ld_or(okb, a.s, kb, 0.0);
    const double da = ld_or(oka, a.dsdh, ka, 0.0), db = ld_or(okb, a.dsdh, kb, 0.0);
    const double aa = ld_or(oka, a.acc, ka, 0.0), ab = ld_or(okb, a.acc, kb, 0.0);
    const double ma = ld_or(oka, a.mel, ka, 0.0), mb = ld_or(okb, a.mel, kb, 0.0);
    const double h = (v ? a.hv : a.hu)[tt], s = (v ? a.sv : a.su)[tt], f3 = (v ? a.f3v : a.f3u)[tt];
    double *out = v ? a.bv : a.bu;
    if (!inner) {
        out[tt] = 0.0;
        return;
    }
    const double rd = v ? a.rdy : a.rdx;
    // the surface adjusted for the implicit step, s + theta dt dsdh (a - m),
    // on the two cells (0 off the mask)
    double a1 = okb ? (hb ? sb + (a.tdt * db) * (ab - mb) : 0.0) : 0.0;
    double a0 = oka ? (ha ? sa + (a.tdt * da) * (aa - ma) : 0.0) : 0.0;
    double ts = rd * a1 - rd * a0;
    double f1 = (rg * h) * ts;
    double m1 = okb ? (hb ? 1.0 : 0.0) : 0.0;
    double m0 = oka ? (ha ? 1.0 : 0.0) : 0.0;
    double tm = rd * m1 - rd * m0;
    double d = h - (s - a.sl);
    if (!(d > 0.0)) d = 0.0;
    double X = (hri * (h * h) - hrw * (d * d)) - (a.ri * h) * s;
    double f2 = (tm * a.g) * X;
    out[tt] = (f1 + f2) + (-f3);
}

// ===========================================================================
// Operator application, residual, diagonal, colour sweeps.

// diag(A) at inner points: the stencil evaluated on a unit vector, which is
// what get_op_diag's colour probes (update_preconditioners.jl:92-109) see.
template <typename T>
__global__ void k_diag(GridDims g, OpCoef<T> c, T *du, T *dv)
{
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int nu = g.nxu * g.nyu, nv = g.nxv * g.nyv;
    if (t < nu) {
        int i = t % g.nxu, j = t / g.nxu;
        DeltaIn<T> in{i, j, 0};
        du[t] = c.ui[t] ? op_u(c, in, i, j) : T(0);
    } else if (t < nu + nv) {
        int tv = t - nu;
        int i = tv % g.nxv, j = tv / g.nxv;
        DeltaIn<T> in{i, j, 1};
        dv[tv] = c.vi[tv] ? op_v(c, in, i, j) : T(0);
    }
}

// ===========================================================================
// Haar transforms on 16x16 tiles in LDS.  dir: 0 forward, 1 inverse,
// 2 transposed inverse.  y factor first, then x (the order KroneckerProduct
// mul! takes for square factors); each output sums its terms in increasing
// source index.

// One composed row of a table-driven transform: sum over the row's n terms
// of coef * src[col * stride], in the table's order.  The row's whole table
// entries are loaded first (MAX_HAAR_NNZ of each; those past n are not used),
// so that a term waits on its LDS read only, not on two table loads.
template <typename T>
__device__ __forceinline__ T haar_table_row(const HaarTable *tab, int dir, int m, int r, const T *src, int stride)
{
    const int n = tab->nnz[dir][m][r];
    float cf[MAX_HAAR_NNZ];
    int cl[MAX_HAAR_NNZ];
#pragma unroll
    for (int q = 0; q < MAX_HAAR_NNZ; ++q) {
        cf[q] = tab->coef[dir][m][r][q];
        cl[q] = tab->col[dir][m][r][q];
    }
    T acc = T(0);
#pragma unroll
    for (int q = 0; q < MAX_HAAR_NNZ; ++q)
        if (q < n) acc = acc + (T)cf[q] * src[cl[q] * stride];
    return acc;
}

template <typename T>
__device__ __forceinline__ void haar_tile(const HaarTable *tab, int dir, T (*tile)[TILE + 1], T (*tmp)[TILE + 1],
                                          int i0, int j0, int nxw, int nyw)
{
    const int lx = threadIdx.x & 15, ly = threadIdx.x >> 4;
    const int B = tab->B;
    const int i = i0 + lx, j = j0 + ly;
    // y pass
    if (i < nxw && j < nyw) {
        int jb = ly - (ly % B);
        int m = nyw - (j0 + jb);
        m = m < B ? m : B;
        int r = ly - jb;
        tmp[ly][lx] = haar_table_row<T>(tab, dir, m, r, &tile[jb][lx], TILE + 1);
    }
    __syncthreads();
    // x pass, with the transposed element mapping of the y pass swapped (the
    // lanes of a wave share the column, so rows of one length)
    const int lyx = threadIdx.x & 15, lxx = threadIdx.x >> 4;
    if (i0 + lxx < nxw && j0 + lyx < nyw) {
        int ib = lxx - (lxx % B);
        int m = nxw - (i0 + ib);
        m = m < B ? m : B;
        int r = lxx - ib;
        tile[lyx][lxx] = haar_table_row<T>(tab, dir, m, r, &tmp[lyx][ib], 1);
    }
    __syncthreads();
}

// update_wavelets! (src/Wavelets/update_wavelets.jl:6-32): dwt of the masked
// velocities, threshold mask, zero warm start.
__global__ void k_tile_wavelets(GridDims g, const HaarTable *tab, const double *U, const double *V,
                                const uint8_t *um, const uint8_t *vm, double *Wu, double *Wv,
                                uint8_t *mwu, uint8_t *mwv, double *cu, double *cv, double thr)
{
    __shared__ double tile[TILE][TILE + 1];
    __shared__ double tmp[TILE][TILE + 1];
    const int lx = threadIdx.x & 15, ly = threadIdx.x >> 4;
    const int bx = blockIdx.x, by = blockIdx.y;
    const int i0 = bx * TILE, j0 = by * TILE;
    const int i = i0 + lx, j = j0 + ly;
    if (bx < g.nbxu && by < g.nbyu) {
        int k = i + g.nxu * j;
        bool ok = i < g.nxu && j < g.nyu;
        const double x = ld_or(ok, U, k, 0.0);
        tile[ly][lx] = (ld_or(ok, um, k, (uint8_t)0) != 0) ? x : 0.0;
        __syncthreads();
        haar_tile<double>(tab, 0, tile, tmp, i0, j0, g.nxu, g.nyu);
        if (ok) {
            double w = tile[ly][lx];
            Wu[k] = w;
            mwu[k] = fabs(w) >= thr ? 1 : 0;
            cu[k] = 0.0;
        }
        __syncthreads();
    }
    if (bx < g.nbxv && by < g.nbyv) {
        int k = i + g.nxv * j;
        bool ok = i < g.nxv && j < g.nyv;
        const double x = ld_or(ok, V, k, 0.0);
        tile[ly][lx] = (ld_or(ok, vm, k, (uint8_t)0) != 0) ? x : 0.0;
        __syncthreads();
        haar_tile<double>(tab, 0, tile, tmp, i0, j0, g.nxv, g.nyv);
        if (ok) {
            double w = tile[ly][lx];
            Wv[k] = w;
            mwv[k] = fabs(w) >= thr ? 1 : 0;
            cv[k] = 0.0;
        }
        __syncthreads();
    }
}

// ===========================================================================
// Haar transforms with +-1 coefficients: the inverse P and its transpose R.

// P's rows as bit masks (k_coarse_diag): bit c of `nz` marks a term in column
// c and bit c of `neg` its sign, one table per `levels` (0..3).
struct HaarMasks {
    uint16_t nz[17][16];
    uint16_t neg[17][16];
};
__constant__ HaarMasks c_haar[4];

// acc + v or acc - v (neg), with the sign as an exact factor: one instruction,
// rounded as the addition.
__device__ __forceinline__ double add_sign(double acc, double v, bool neg) { return __builtin_fma(neg ? -1.0 : 1.0, v, acc); }
__device__ __forceinline__ float add_sign(float acc, float v, bool neg) { return __builtin_fmaf(neg ? -1.0f : 1.0f, v, acc); }

// One 16-point line of P, the composed inverse of wavelet_matrix
// (src/Wavelets/update_wavelets.jl:38-89) with blocks of B = 2^(LEV+1)
// points: y_i = sum over c of P[i][c] x_c, the terms added in increasing
// column order as the oracle adds them.  Row i has the block's column 0 and
// one column e_h = o + h per pair (o, e_h) that i belongs to, h = 1 .. B/2: +1
// where i is on the pair's upper half (bit h of i set), else -1.  In
// increasing order these are the e_h of the set bits, then of the clear ones.
// A thread computes rows 2w and 2w + 1 of the half line `half` (8 points): the
// two rows share all columns and differ in one sign.  With LEV = 3 the block
// is the whole line: its columns 0 and 8 come first in the second half (x_0 +
// x_8), and in the first half x_0 first and -x_8 last.  w is uniform over a
// wavefront, so columns and signs are, and the wavefronts share one code;
// load and rows are apart so that the operands of several lines can be in
// flight.  Points past the end of the grid must hold zero: their terms then
// change nothing, which leaves wavelet_matrix's partial blocks.
template <int LEV, typename T>
struct HaarLineP {
    static constexpr int S = LEV < 2 ? LEV + 1 : 3;  // columns of a row inside the half line
    T base, x8, v[S];
    __device__ __forceinline__ void load(const T *src, int st, int half, int w)
    {
        const T *z = src + 8 * half * st;
        x8 = T(0);
        if constexpr (LEV == 0) {
            base = z[2 * w * st];
            v[0] = z[(2 * w + 1) * st];
        } else if constexpr (LEV == 1) {
            const int o = 2 * (w & 2);
            base = z[o * st];
            v[0] = z[(o + 1 + (w & 1)) * st];
            v[1] = z[(o + 2 + (w & 1)) * st];
        } else {
            // columns by w: 1 2 4, 2 3 4, 4 5 6, 4 6 7
            const int k0 = w == 0 ? 1 : (w == 1 ? 2 : 4);
            const int k1 = w == 0 ? 2 : (w == 1 ? 3 : (w == 2 ? 5 : 6)), k2 = w < 2 ? 4 : (w == 2 ? 6 : 7);
            base = LEV == 3 ? src[0] : z[0];
            if constexpr (LEV == 3) x8 = src[8 * st];
            v[0] = z[k0 * st];
            v[1] = z[k1 * st];
            v[2] = z[k2 * st];
        }
    }
    __device__ __forceinline__ void rows(T *dst, int st, int half, int w) const
    {
        T b = base, tail = T(0);
        if constexpr (LEV == 3) {
            b = half ? b + x8 : b;
            tail = half ? T(0) : x8;
        }
        const int plus = LEV == 0 ? 0 : (LEV == 1 ? (w & 1) : (w & 1) + (w >> 1));  // + signs of row 2w
        T lo = b, hi = b;
#pragma unroll
        for (int k = 0; k < S; ++k) {
            lo = add_sign(lo, v[k], k >= plus);
            hi = add_sign(hi, v[k], k >= plus + 1);
        }
        if constexpr (LEV == 3) {
            lo = lo - tail;
            hi = hi - tail;
        }
        T *d = dst + (8 * half + 2 * w) * st;
        d[0] = lo;
        d[st] = hi;
    }
};

template <int LEV, typename T>
__device__ __forceinline__ void haar_line_P(const T *src, T *dst, int st, int half, int w)
{
    HaarLineP<LEV, T> p;
    p.load(src, st, half, w);
    p.rows(dst, st, half, w);
}

// One 16-point line of R = P^T: row o + h of a pair is -1 on the h points
// from o and +1 on the h points from o + h, row 0 of a block sums the block;
// terms in increasing order.  A row's leading minus terms are the negated
// prefix sum of its points, the same roundings as subtracting them one by
// one, so the long rows share their prefixes.  The four wavefronts take the
// block sums (LEV = 3: rows 0 and 8, one per half), the rows 4 and 12, the
// rows 2 and 6 of each half, and the odd rows; a thread of the first adds
// 16 terms, of the others at most 8.
template <int LEV, typename T>
__device__ __forceinline__ void haar_line_R(const T *src, T *dst, int st, int half, int w)
{
    const T *z = src + 8 * half * st;
    T *d = dst + 8 * half * st;
    if (w == 0) {
        if constexpr (LEV == 3) {
            T x[16];
#pragma unroll
            for (int c = 0; c < 16; ++c) x[c] = src[c * st];
            T a = x[0];
#pragma unroll
            for (int c = 1; c < 8; ++c) a = a + x[c];
            a = half ? -a : a;
#pragma unroll
            for (int c = 8; c < 16; ++c) a = a + x[c];
            d[0] = a;
        } else {
            T x[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) x[c] = z[c * st];
            constexpr int B = 2 << LEV;
#pragma unroll
            for (int o = 0; o < 8; o += B) {
                T a = x[o];
#pragma unroll
                for (int c = 1; c < B; ++c) a = a + x[o + c];
                d[o * st] = a;
            }
        }
    } else if (w == 1) {
        if constexpr (LEV >= 2) {
            T x[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) x[c] = z[c * st];
            const T a = ((x[0] + x[1]) + x[2]) + x[3];
            d[4 * st] = (((x[4] - a) + x[5]) + x[6]) + x[7];
        }
    } else if (w == 2) {
        if constexpr (LEV >= 1) {
            T x[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) x[c] = z[c * st];
            d[2 * st] = (x[2] - (x[0] + x[1])) + x[3];
            d[6 * st] = (x[6] - (x[4] + x[5])) + x[7];
        }
    } else {
#pragma unroll
        for (int o = 0; o < 8; o += 2) {
            const T a = z[o * st], b = z[(o + 1) * st];
            d[(o + 1) * st] = b - a;
        }
    }
}

// A u tile and a v tile side by side, as the transforms read them.
template <typename T>
using TilePair = T[2][TILE][TILE + 1];

// P (R = false) or R of the u and the v tile of one block, in place, with m
// as scratch: the y lines, then the x lines (the order KroneckerProduct mul!
// takes for square factors).  Every wavefront covers all 32 lines of both
// tiles, a half line per lane, and takes its own rows of each line, so the
// code of a wavefront is straight and the operands of a row are read from
// LDS once, all before the first is used.  The rows as bit masks walked term
// by term (one row per thread, 16 dependent LDS reads in the longest)
// cost the operator's launch 9,200 of its 16,600 cycles on a lone tile.
// Points past the grid's end must hold zero.  Ends with a barrier.
template <bool R, int LEV, typename T>
__device__ __forceinline__ void haar_pair_lev(TilePair<T> &t, TilePair<T> &m)
{
    const int l = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = l & 15, comp = (l >> 4) & 1, half = l >> 5;
    if constexpr (R)
        haar_line_R<LEV, T>(&t[comp][0][q], &m[comp][0][q], TILE + 1, half, w);
    else
        haar_line_P<LEV, T>(&t[comp][0][q], &m[comp][0][q], TILE + 1, half, w);
    __syncthreads();
    if constexpr (R)
        haar_line_R<LEV, T>(&m[comp][q][0], &t[comp][q][0], 1, half, w);
    else
        haar_line_P<LEV, T>(&m[comp][q][0], &t[comp][q][0], 1, half, w);
    __syncthreads();
}

template <bool R, typename T>
__device__ __forceinline__ void haar_pair(int levels, TilePair<T> &t, TilePair<T> &m)
{
    if (levels == 3)
        haar_pair_lev<R, 3, T>(t, m);
    else if (levels == 2)
        haar_pair_lev<R, 2, T>(t, m);
    else if (levels == 1)
        haar_pair_lev<R, 1, T>(t, m);
    else
        haar_pair_lev<R, 0, T>(t, m);
}

// ===========================================================================
// The operator on one 16x16 tile of u and v outputs, every intermediate
// computed once per tile in LDS.  U and V are staged with a one-point halo
// (18 x 18, s.U[y][x] = U(i0-1+x, j0-1+y)); r_xx, r_yy and the implicit
// term on the 17 x 17 h cells and r_xy on the 17 x 17 c corners starting one
// point before the tile.  Arithmetic is that of op_u / op_v (same expressions,
// same order, absent terms zero), so results are bit-identical.
template <typename T>
struct OpTile {
    T U[18][19];
    T V[18][19];
    T rxx[17][18];
    T ryy[17][18];
    T ext[17][18];
    T rxy[17][18];
};

// Coefficients of one h cell and its c corner (the cell (i0-1+x, j0-1+y) of
// the 17 x 17 window, q = x + 17 y), loaded before they are needed so that a
// tile costs one round trip to memory.
template <typename T>
struct CellCoef {
    T heta, dimp, hu0, hu1, hv0, hv1, hetac;
    uint8_t hm, um0, um1, vm0, vm1, cm;
    bool cell, corner;
};

// Coefficients of h cell (a, b) and its c corner; in_window = false leaves
// both absent.
template <typename T>
__device__ __forceinline__ void cell_prefetch_at(const GridDims &g, const OpCoef<T> &c, int a, int b,
                                                 bool in_window, CellCoef<T> &cc)
{
    const int nx = g.nx, ny = g.ny, nxu = g.nxu;
    cc.cell = in_window && a >= 0 && a < nx && b >= 0 && b < ny;
    cc.corner = in_window && a >= 0 && a < nx - 1 && b >= 0 && b < ny - 1;
    // loads issued unconditionally (ld_or); absent entries are never read
    {
        const bool ok = cc.cell;
        const int k = a + nx * b, ku0 = a + nxu * b, kv0 = a + nx * b, kv1 = kv0 + nx;
        cc.hm = ld_or(ok, c.hm, k, (uint8_t)0);
        cc.heta = ld_or(ok, c.heta_h, k, T(0));
        cc.dimp = ld_or(ok, c.dimp, k, T(0));
        cc.um0 = ld_or(ok, c.um, ku0, (uint8_t)0);
        cc.um1 = ld_or(ok, c.um, ku0 + 1, (uint8_t)0);
        cc.hu0 = ld_or(ok, c.hu, ku0, T(0));
        cc.hu1 = ld_or(ok, c.hu, ku0 + 1, T(0));
        cc.vm0 = ld_or(ok, c.vm, kv0, (uint8_t)0);
        cc.vm1 = ld_or(ok, c.vm, kv1, (uint8_t)0);
        cc.hv0 = ld_or(ok, c.hv, kv0, T(0));
        cc.hv1 = ld_or(ok, c.hv, kv1, T(0));
    }
    {
        const int kc = a + (nx - 1) * b;
        cc.cm = ld_or(cc.corner, c.cm, kc, (uint8_t)0);
        cc.hetac = ld_or(cc.corner, c.heta_c, kc, T(0));
    }
}

template <typename T>
__device__ __forceinline__ void cell_prefetch(const GridDims &g, const OpCoef<T> &c, int i0, int j0, int q,
                                              CellCoef<T> &cc)
{
    cell_prefetch_at(g, c, i0 - 1 + q % 17, j0 - 1 + q / 17, q < 289, cc);
}

// Intermediates of the cell / corner at (x, y) of a staged window whose
// points U[y][x] and cells share one origin (same expressions as op_rxx,
// op_ryy, op_extra, op_rxy).
template <typename T, class S>
__device__ __forceinline__ void cell_eval(const OpCoef<T> &c, const CellCoef<T> &cc, int x, int y, S &s)
{
    T rxx = T(0), ryy = T(0), ext = T(0), rxy = T(0);
    if (cc.cell) {
        const T u0 = s.U[y][x], u1 = s.U[y][x + 1], v0 = s.V[y][x], v1 = s.V[y + 1][x];
        if (cc.hm) {
            const T dudx = c.rdx * u1 - c.rdx * u0;
            const T dvdy = c.rdy * v1 - c.rdy * v0;
            rxx = T(2) * (cc.heta * (T(2) * dudx + dvdy));
            ryy = T(2) * (cc.heta * (T(2) * dvdy + dudx));
        }
        const T qx1 = cc.um1 ? cc.hu1 * u1 : T(0);
        const T qx0 = cc.um0 ? cc.hu0 * u0 : T(0);
        const T qy1 = cc.vm1 ? cc.hv1 * v1 : T(0);
        const T qy0 = cc.vm0 ? cc.hv0 * v0 : T(0);
        const T divq = (c.rdx * qx1 - c.rdx * qx0) + (c.rdy * qy1 - c.rdy * qy0);
        ext = cc.dimp * divq;
    }
    if (cc.corner && cc.cm) {
        const T dudy = c.rdy * s.U[y + 1][x + 1] - c.rdy * s.U[y][x + 1];
        const T dvdx = c.rdx * s.V[y + 1][x + 1] - c.rdx * s.V[y + 1][x];
        rxy = cc.hetac * (dudy + dvdx);
    }
    s.rxx[y][x] = rxx;
    s.ryy[y][x] = ryy;
    s.ext[y][x] = ext;
    s.rxy[y][x] = rxy;
}

template <typename T>
__device__ __forceinline__ void cell_compute(const OpCoef<T> &c, const CellCoef<T> &cc, int q, OpTile<T> &s)
{
    if (q >= 289) return;
    cell_eval(c, cc, q % 17, q / 17, s);
}

// Coefficients of the thread's own u and v output points.
template <typename T>
struct PointCoef {
    T bu, hu, bv, hv;
    bool oku, okv, ui, um, vi, vm;
    int ku, kv;
};

// fx at the u point (i0 + x, j0 + y), whose value is s.U[y + 1][x + 1] and
// whose cell (i, j) is s.rxx[y + 1][x + 1]
template <typename T, class S>
__device__ __forceinline__ T optile_u(const OpCoef<T> &c, const S &s, const PointCoef<T> &pc, int x, int y)
{
    const T d_rxx_dx = c.rdx * s.rxx[y + 1][x + 1] - c.rdx * s.rxx[y + 1][x];
    const T d_rxy_dy = c.rdy * s.rxy[y + 1][x] - c.rdy * s.rxy[y][x];
    const T taubx = pc.um ? pc.bu * s.U[y + 1][x + 1] : T(0);
    const T d_extra_dx = c.rdx * s.ext[y + 1][x + 1] - c.rdx * s.ext[y + 1][x];
    return ((d_rxx_dx + d_rxy_dy) - taubx) - pc.hu * d_extra_dx;
}

// fy at the v point (i0 + x, j0 + y), with the same window convention
template <typename T, class S>
__device__ __forceinline__ T optile_v(const OpCoef<T> &c, const S &s, const PointCoef<T> &pc, int x, int y)
{
    const T d_ryy_dy = c.rdy * s.ryy[y + 1][x + 1] - c.rdy * s.ryy[y][x + 1];
    const T d_rxy_dx = c.rdx * s.rxy[y][x + 1] - c.rdx * s.rxy[y][x];
    const T tauby = pc.vm ? pc.bv * s.V[y + 1][x + 1] : T(0);
    const T d_extra_dy = c.rdy * s.ext[y + 1][x + 1] - c.rdy * s.ext[y][x + 1];
    return ((d_ryy_dy + d_rxy_dx) - tauby) - pc.hv * d_extra_dy;
}

// The operator on a tile of u and v outputs from global memory.  What bounds
// these kernels on any grid is the number of load and LDS instructions of a
// wavefront, so each operand is loaded once: a thread loads its own u and v
// point (value, thickness, drag, mask bits) and its own h cell and corner;
// wavefront 3 adds the 64 points of the four sides of the one-point halo,
// wavefront 2 the two halo corners that are read (u at (16, -1), v at
// (-1, 16)), wavefront 0 the 33 cells before the tile.  15 to 21 loads a
// wavefront instead of 42 with the window walked by 256 threads and every
// cell loading its four thicknesses and six masks.  The fluxes h u and h v
// of the implicit term are formed once per point, masked, and staged.
// The arithmetic and the masks are those of op_u / op_v: what lies off a mask
// is selected away, not multiplied by a zero coefficient, so that a value that
// is not finite there (missing data outside the ice) reaches no output.

// Mask bits of a u or v point: 1 inner, 2 u / v mask, 4 wavelet mask.
enum { MB_INNER = 1, MB_POINT = 2, MB_WAVELET = 4 };

// ... from the separate masks (mw may be null: bit 4 clear)
template <bool MW>
struct MaskSep {
    const uint8_t *ui, *um, *vi, *vm, *mwu, *mwv;
    __device__ __forceinline__ unsigned u(bool ok, int k) const
    {
        const int q = ok ? k : 0;
        const unsigned a = ui[q], b = um[q], w = MW ? mwu[q] : 0;
        return ok ? (a ? MB_INNER : 0u) | (b ? MB_POINT : 0u) | (w ? MB_WAVELET : 0u) : 0u;
    }
    __device__ __forceinline__ unsigned v(bool ok, int k) const
    {
        const int q = ok ? k : 0;
        const unsigned a = vi[q], b = vm[q], w = MW ? mwv[q] : 0;
        return ok ? (a ? MB_INNER : 0u) | (b ? MB_POINT : 0u) | (w ? MB_WAVELET : 0u) : 0u;
    }
};

// The coarse values around a tile from which k_cg_step forms P u on the
// halo (LEV + 2 lines per side, haar_halo_offset; 5 at three levels).
template <typename T>
struct HaloLds {
    T x[2][10][17];   // component; columns left (0..4) and right (5..9), by y
    T y[2][10][16];   // rows below (0..4) and above (5..9), by x
    T c[2][5][5];     // the corner block, [y][x]
    T lx[2][10][17];  // y sums of x
    T ly[2][2][16];   // y sums of y: rows -1 and 16, by x
    T lc[2][5];       // y sums of c
};

// Window point (x, y) is (i0 - 1 + x, j0 - 1 + y); cell (x, y) has the same
// origin.  The window's room also holds the tiles of R (h; the window is
// read last before the barrier that the outputs follow) and, before it, the
// coarse halo (n); the cells' room holds the tiles of P (p) before them.
template <typename T>
struct OpLds {
    union {
        struct {
            T U[18][19], V[18][19], QX[18][19], QY[18][19];
        } w;
        struct {
            TilePair<T> t, m;
        } h;
        HaloLds<T> n;
    };
    union {
        struct {
            T rxx[17][18], ryy[17][18], ext[17][18], rxy[17][18];
        };
        struct {
            TilePair<T> t, m;
        } p;
    };
};

// Intermediates of one cell.
template <typename T>
struct OpCell {
    T rxx, ryy, ext, rxy;
    __device__ __forceinline__ void store(OpLds<T> &s, int x, int y) const
    {
        s.rxx[y][x] = rxx;
        s.ryy[y][x] = ryy;
        s.ext[y][x] = ext;
        s.rxy[y][x] = rxy;
    }
};

// What a thread holds of its tile.  The thicknesses and drags are zero off the
// u and v masks (an inner point is on its mask).
template <typename T>
struct OpOwn {
    T u, v, hu, hv, bu, bv;
    T heta, dimp, hetac;
    OpCell<T> cell;   // the intermediates of its cell
    unsigned mu, mv;  // mask bits
    unsigned mc;      // ... of its cell (CELL_*)
    bool oku, okv;
    int ku, kv;
};

// Mask bits of a cell: 1 on the grid, 2 h mask, 4 its corner on the c mask.
enum { CELL_GRID = 1, CELL_H = 2, CELL_CORNER = 4 };

// h cell (a, b) and its corner: 0 outside their grids.  Returns the mask bits.
template <typename T>
__device__ __forceinline__ unsigned op_cell_load(const GridDims &g, const OpCoef<T> &c, int a, int b, T &heta, T &dimp,
                                                 T &hetac)
{
    const bool cell = a >= 0 && a < g.nx && b >= 0 && b < g.ny;
    const bool corner = a >= 0 && a < g.nx - 1 && b >= 0 && b < g.ny - 1;
    heta = ld_or(cell, c.heta_h, a + g.nx * b, T(0));
    dimp = ld_or(cell, c.dimp, a + g.nx * b, T(0));
    hetac = ld_or(corner, c.heta_c, a + (g.nx - 1) * b, T(0));
    const uint8_t hm = ld_or(cell, c.hm, a + g.nx * b, (uint8_t)0);
    const uint8_t cm = ld_or(corner, c.cm, a + (g.nx - 1) * b, (uint8_t)0);
    return (cell ? CELL_GRID : 0u) | (hm ? CELL_H : 0u) | (cm ? CELL_CORNER : 0u);
}

// Intermediates of cell (x, y) (the expressions of op_rxx, op_ryy, op_extra,
// op_rxy).  Cell (0, 0) reads one absent window point of each kind and corner
// (16, 16) another; no output reads what they feed.
// u, v, qx, qy: the window at (x, y).  MASKED: by the cell's mask bits mc;
// else its coefficients are zero off the masks and the window is finite there.
template <bool MASKED, typename T>
__device__ __forceinline__ OpCell<T> op_cell(T rdx, T rdy, const OpLds<T> &s, int x, int y, T u, T v, T qx, T qy,
                                             T heta, T dimp, T hetac, unsigned mc)
{
    const T u1 = s.w.U[y][x + 1], v1 = s.w.V[y + 1][x];
    const T dudx = rdx * u1 - rdx * u;
    const T dvdy = rdy * v1 - rdy * v;
    const T divq = (rdx * s.w.QX[y][x + 1] - rdx * qx) + (rdy * s.w.QY[y + 1][x] - rdy * qy);
    const T dudy = rdy * s.w.U[y + 1][x + 1] - rdy * u1;
    const T dvdx = rdx * s.w.V[y + 1][x + 1] - rdx * v1;
    OpCell<T> r{T(2) * (heta * (T(2) * dudx + dvdy)), T(2) * (heta * (T(2) * dvdy + dudx)), dimp * divq, hetac * (dudy + dvdx)};
    if constexpr (MASKED) {
        r.rxx = (mc & CELL_H) ? r.rxx : T(0);
        r.ryy = (mc & CELL_H) ? r.ryy : T(0);
        r.ext = (mc & CELL_GRID) ? r.ext : T(0);
        r.rxy = (mc & CELL_CORNER) ? r.rxy : T(0);
    }
    return r;
}

// Halo points a thread stages: u at (ux, uy) and v at (vx, vy) of the window.
// op_halo_sides: wavefront 3 the four sides, wavefront 2 the corners.
struct HaloPos {
    int ux, uy, vx, vy;
    bool hu, hv;  // holds a u / a v halo point
};

// Side point l (0..63: left and right columns by y, bottom and top rows by x)
__device__ __forceinline__ void halo_side(int l, int &x, int &y)
{
    const int q = 1 + (l & 15), far = (l & 16) ? 17 : 0;
    x = l < 32 ? far : q;
    y = l < 32 ? q : far;
}

__device__ __forceinline__ HaloPos op_halo_sides(int w, int l)
{
    HaloPos h{17, 0, 0, 17, w == 3 || (w == 2 && l == 0), w == 3 || (w == 2 && l == 0)};
    if (w == 3) {
        halo_side(l, h.ux, h.uy);
        h.vx = h.ux;
        h.vy = h.uy;
    }
    return h;
}

// Coefficients of a tile besides its points' values: the thread's own point
// and cell, its halo points' thicknesses (zero off the masks), and the cell
// before the tile that it computes (wavefront 0, lanes 0..32: (0, 0..16), (1..16, 0)).
template <typename T>
struct OpCoefRegs {
    T hhu, hhv;
    bool hmu, hmv;    // the halo points are on the u, v mask
    T eh, ed, ec;
    unsigned em;      // the cell's mask bits
    int ex, ey;
};

// ... and where that cell is
template <typename T>
__device__ __forceinline__ void op_extra_cell(int l, OpCoefRegs<T> &r)
{
    r.ex = l < 17 ? 0 : (l < 33 ? l - 16 : 16);
    r.ey = l < 17 ? l : 0;
    r.eh = r.ed = r.ec = T(0);
    r.em = 0;
}

template <typename T, class M>
__device__ __forceinline__ void op_coef_load(const GridDims &g, const OpCoef<T> &c, const M &mask, int i0, int j0,
                                             const HaloPos &h, bool halo_wave, OpOwn<T> &o, OpCoefRegs<T> &r)
{
    const int lx = threadIdx.x & 15, ly = threadIdx.x >> 4, l = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const T ohu = ld_or(o.oku, c.hu, o.ku, T(0)), ohv = ld_or(o.okv, c.hv, o.kv, T(0));
    r.hhu = r.hhv = T(0);
    r.hmu = r.hmv = false;
    if (halo_wave) {
        const int iu = i0 - 1 + h.ux, ju = j0 - 1 + h.uy, iv = i0 - 1 + h.vx, jv = j0 - 1 + h.vy;
        const bool oku = h.hu && iu >= 0 && iu < g.nxu && ju >= 0 && ju < g.nyu;
        const bool okv = h.hv && iv >= 0 && iv < g.nxv && jv >= 0 && jv < g.nyv;
        const T u = ld_or(oku, c.hu, iu + g.nxu * ju, T(0)), v = ld_or(okv, c.hv, iv + g.nxv * jv, T(0));
        r.hmu = mask.u(oku, iu + g.nxu * ju) & MB_POINT;
        r.hmv = mask.v(okv, iv + g.nxv * jv) & MB_POINT;
        r.hhu = r.hmu ? u : T(0);
        r.hhv = r.hmv ? v : T(0);
    }
    o.mc = op_cell_load(g, c, i0 + lx, j0 + ly, o.heta, o.dimp, o.hetac);
    op_extra_cell(l, r);
    if (w == 0) r.em = op_cell_load(g, c, i0 - 1 + r.ex, j0 - 1 + r.ey, r.eh, r.ed, r.ec);
    const T obu = ld_or(o.oku, c.bu, o.ku, T(0)), obv = ld_or(o.okv, c.bv, o.kv, T(0));
    o.hu = (o.mu & MB_POINT) ? ohu : T(0);
    o.hv = (o.mv & MB_POINT) ? ohv : T(0);
    o.bu = (o.mu & MB_POINT) ? obu : T(0);
    o.bv = (o.mv & MB_POINT) ? obv : T(0);
}

// Stage the window (the thread's own point and its halo points hu, hv) and
// compute the cells' intermediates.  Ends with a barrier, after which the
// window is free.  MASKED: o and r hold the mask bits (op_coef_load).
template <bool MASKED, typename T>
__device__ __forceinline__ void op_cells(T rdx, T rdy, const HaloPos &h, T hu, T hv, OpOwn<T> &o,
                                         const OpCoefRegs<T> &r, OpLds<T> &s)
{
    const int lx = threadIdx.x & 15, ly = threadIdx.x >> 4;
    s.w.U[ly + 1][lx + 1] = o.u;
    s.w.V[ly + 1][lx + 1] = o.v;
    T qx = o.hu * o.u, qy = o.hv * o.v;
    if constexpr (MASKED) {
        qx = (o.mu & MB_POINT) ? qx : T(0);
        qy = (o.mv & MB_POINT) ? qy : T(0);
    }
    s.w.QX[ly + 1][lx + 1] = qx;
    s.w.QY[ly + 1][lx + 1] = qy;
    if (h.hu) {
        s.w.U[h.uy][h.ux] = hu;
        s.w.QX[h.uy][h.ux] = !MASKED || r.hmu ? r.hhu * hu : T(0);
    }
    if (h.hv) {
        s.w.V[h.vy][h.vx] = hv;
        s.w.QY[h.vy][h.vx] = !MASKED || r.hmv ? r.hhv * hv : T(0);
    }
    __syncthreads();
    o.cell = op_cell<MASKED>(rdx, rdy, s, lx + 1, ly + 1, o.u, o.v, qx, qy, o.heta, o.dimp, o.hetac, o.mc);
    if (__builtin_amdgcn_readfirstlane(threadIdx.x) == 0) {
        // lanes past the 33 cells before the tile repeat the last
        const OpCell<T> first = op_cell<MASKED>(rdx, rdy, s, r.ex, r.ey, s.w.U[r.ey][r.ex], s.w.V[r.ey][r.ex],
                                                s.w.QX[r.ey][r.ex], s.w.QY[r.ey][r.ex], r.eh, r.ed, r.ec, r.em);
        first.store(s, r.ex, r.ey);
    }
    o.cell.store(s, lx + 1, ly + 1);
    __syncthreads();
}

__device__ __forceinline__ void op_own_index(const GridDims &g, int i, int j, bool &oku, bool &okv, int &ku, int &kv)
{
    oku = i < g.nxu && j < g.nyu;
    okv = i < g.nxv && j < g.nyv;
    ku = i + g.nxu * j;
    kv = i + g.nxv * j;
}

// Load the tile of (xu, xv) and its coefficients and compute the cells'
// intermediates.
template <typename T, class M>
__device__ __forceinline__ void op_tile(const GridDims &g, const OpCoef<T> &c, const M &mask, const T *xu, const T *xv,
                                        int i0, int j0, OpLds<T> &s, OpOwn<T> &o)
{
    const int l = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    op_own_index(g, i0 + (threadIdx.x & 15), j0 + (threadIdx.x >> 4), o.oku, o.okv, o.ku, o.kv);
    o.u = ld_or(o.oku, xu, o.ku, T(0));
    o.v = ld_or(o.okv, xv, o.kv, T(0));
    o.mu = mask.u(o.oku, o.ku);
    o.mv = mask.v(o.okv, o.kv);
    const HaloPos h = op_halo_sides(w, l);
    T hu = T(0), hv = T(0);
    if (w >= 2) {
        const int iu = i0 - 1 + h.ux, ju = j0 - 1 + h.uy, iv = i0 - 1 + h.vx, jv = j0 - 1 + h.vy;
        hu = ld_or(h.hu && iu >= 0 && iu < g.nxu && ju >= 0 && ju < g.nyu, xu, iu + g.nxu * ju, T(0));
        hv = ld_or(h.hv && iv >= 0 && iv < g.nxv && jv >= 0 && jv < g.nyv, xv, iv + g.nxv * jv, T(0));
    }
    OpCoefRegs<T> r;
    op_coef_load(g, c, mask, i0, j0, h, w >= 2, o, r);
    op_cells<true>(c.rdx, c.rdy, h, hu, hv, o, r, s);
}

// A x at the thread's u point and v point (inner or not)
template <typename T>
__device__ __forceinline__ T op_out_u(T rdx, T rdy, const OpLds<T> &s, const OpOwn<T> &o)
{
    const int x = threadIdx.x & 15, y = threadIdx.x >> 4;
    const T d_rxx_dx = rdx * o.cell.rxx - rdx * s.rxx[y + 1][x];
    const T d_rxy_dy = rdy * s.rxy[y + 1][x] - rdy * s.rxy[y][x];
    const T taubx = o.bu * o.u;
    const T d_extra_dx = rdx * o.cell.ext - rdx * s.ext[y + 1][x];
    return ((d_rxx_dx + d_rxy_dy) - taubx) - o.hu * d_extra_dx;
}

template <typename T>
__device__ __forceinline__ T op_out_v(T rdx, T rdy, const OpLds<T> &s, const OpOwn<T> &o)
{
    const int x = threadIdx.x & 15, y = threadIdx.x >> 4;
    const T d_ryy_dy = rdy * o.cell.ryy - rdy * s.ryy[y][x + 1];
    const T d_rxy_dx = rdx * s.rxy[y][x + 1] - rdx * s.rxy[y][x];
    const T tauby = o.bv * o.v;
    const T d_extra_dy = rdy * o.cell.ext - rdy * s.ext[y][x + 1];
    return ((d_ryy_dy + d_rxy_dx) - tauby) - o.hv * d_extra_dy;
}

// R A x of the tile into s.h.t (A zero off the inner masks; valid at the
// wavelet masks' points), x on the fine grid.  Ends with a barrier.
template <typename T, class M>
__device__ __forceinline__ void op_restrict_tile(const GridDims &g, const OpCoef<T> &c, const M &mask, int levels,
                                                 const T *xu, const T *xv, int i0, int j0, OpLds<T> &s, OpOwn<T> &o)
{
    const int lx = threadIdx.x & 15, ly = threadIdx.x >> 4;
    op_tile(g, c, mask, xu, xv, i0, j0, s, o);
    const T yu = (o.mu & MB_INNER) ? op_out_u(c.rdx, c.rdy, s, o) : T(0), yv = (o.mv & MB_INNER) ? op_out_v(c.rdx, c.rdy, s, o) : T(0);
    s.h.t[0][ly][lx] = yu;
    s.h.t[1][ly][lx] = yv;
    __syncthreads();
    haar_pair<true, T>(levels, s.h.t, s.h.m);
}

// ===========================================================================
// Operator application and residual on 16 x 16 tiles of u and v points: the
// tile stages its inputs with a one-point halo and its coefficients once
// (op_tile), computes every intermediate once, and each thread evaluates its
// u and its v point.  The arithmetic is that of op_u / op_v, so the results
// equal the per-point forms bit for bit.  Launched as nblk workgroups
// (xcd_band_tile).

// Tile (bx, by) of this workgroup in a one-dimensional launch of nblk (a
// multiple of 8) workgroups over an nbx x nby tile grid.  Workgroups are
// dispatched round-robin over the 8 XCDs; workgroup w takes tile
// L = (w % 8) (nblk / 8) + w / 8 of a column-major walk (cols = true: each
// XCD takes a band of whole tile columns, so the halos that vertical and
// horizontal neighbours share mostly stay in its L2) or a row-major one (a
// band of whole tile rows).  Returns false for the padding workgroups.
__device__ __forceinline__ bool xcd_band_tile(int nbx, int nby, int nblk, bool cols, int &bx, int &by)
{
    const int w = blockIdx.x;
    const int L = (w & 7) * (nblk >> 3) + (w >> 3);
    bx = cols ? L / nby : L % nbx;
    by = cols ? L % nby : L / nbx;
    return L < nbx * nby;
}

// The coefficients a tile's own u and v points read (no wavelet masks).
template <typename T>
__device__ __forceinline__ void point_prefetch_op(const GridDims &g, const OpCoef<T> &c, int i, int j, bool has_u,
                                                  bool has_v, PointCoef<T> &pc)
{
    pc.oku = has_u && i < g.nxu && j < g.nyu;
    pc.okv = has_v && i < g.nxv && j < g.nyv;
    pc.ku = i + g.nxu * j;
    pc.kv = i + g.nxv * j;
    // loads issued unconditionally (ld_or)
    pc.ui = ld_or(pc.oku, c.ui, pc.ku, (uint8_t)0) != 0;
    pc.um = ld_or(pc.oku, c.um, pc.ku, (uint8_t)0) != 0;
    pc.bu = ld_or(pc.oku, c.bu, pc.ku, T(0));
    pc.hu = ld_or(pc.oku, c.hu, pc.ku, T(0));
    pc.vi = ld_or(pc.okv, c.vi, pc.kv, (uint8_t)0) != 0;
    pc.vm = ld_or(pc.okv, c.vm, pc.kv, (uint8_t)0) != 0;
    pc.bv = ld_or(pc.okv, c.bv, pc.kv, T(0));
    pc.hv = ld_or(pc.okv, c.hv, pc.kv, T(0));
}

// y = A x at inner points, 0 elsewhere
template <typename T>
__global__ void __launch_bounds__(256) k_op(GridDims g, OpCoef<T> c, const T *xu, const T *xv, T *yu, T *yv,
                                            int nblk)
{
    __shared__ OpLds<T> s;
    int bx, by;
    if (!xcd_band_tile(g.nbx, g.nby, nblk, true, bx, by)) return;
    OpOwn<T> o;
    op_tile(g, c, MaskSep<false>{c.ui, c.um, c.vi, c.vm, nullptr, nullptr}, xu, xv, bx * TILE, by * TILE, s, o);
    if (o.oku) yu[o.ku] = (o.mu & MB_INNER) ? op_out_u(c.rdx, c.rdy, s, o) : T(0);
    if (o.okv) yv[o.kv] = (o.mv & MB_INNER) ? op_out_v(c.rdx, c.rdy, s, o) : T(0);
}

// r = b - A x at inner points (get_resid!, utilities.jl:549-552); per-tile
// partials of sum r^2 into Pr and, if Pb != nullptr, of sum b^2 into Pb (u
// tiles first, then v tiles); if fu != nullptr, r also into fu, fv at the
// inner points (the residual fields of set_residual!,
// update_velocities.jl:428-433; their other points are left as they are).
template <typename T>
__global__ void __launch_bounds__(256) k_tile_resid(GridDims g, OpCoef<T> c, const T *xu, const T *xv, const T *bu,
                                                    const T *bv, T *ru, T *rv, double *Pr, double *Pb, int nblk,
                                                    T *fu = nullptr, T *fv = nullptr)
{
    __shared__ OpLds<T> s;
    __shared__ double lds[8];
    int bx, by;
    if (!xcd_band_tile(g.nbx, g.nby, nblk, true, bx, by)) return;
    const bool has_u = bx < g.nbxu && by < g.nbyu, has_v = bx < g.nbxv && by < g.nbyv;
    // the thread's right-hand side, loaded before the operator's barriers
    const int i = bx * TILE + (threadIdx.x & 15), j = by * TILE + (threadIdx.x >> 4);
    const T b_u = ld_or(i < g.nxu && j < g.nyu, bu, i + g.nxu * j, T(0));
    const T b_v = ld_or(i < g.nxv && j < g.nyv, bv, i + g.nxv * j, T(0));
    OpOwn<T> o;
    op_tile(g, c, MaskSep<false>{c.ui, c.um, c.vi, c.vm, nullptr, nullptr}, xu, xv, bx * TILE, by * TILE, s, o);
    if (has_u) {
        double r2 = 0.0, b2 = 0.0;
        if (o.oku) {
            const T r = (o.mu & MB_INNER) ? b_u - op_out_u(c.rdx, c.rdy, s, o) : T(0);
            ru[o.ku] = r;
            if (fu && (o.mu & MB_INNER)) fu[o.ku] = r;
            r2 = (double)r * (double)r;
            b2 = (double)b_u * (double)b_u;
        }
        tree256x2(r2, b2, lds);
        if (threadIdx.x == 0) {
            Pr[bx + g.nbxu * by] = r2;
            if (Pb) Pb[bx + g.nbxu * by] = b2;
        }
    }
    if (has_v) {
        double r2 = 0.0, b2 = 0.0;
        if (o.okv) {
            const T r = (o.mv & MB_INNER) ? b_v - op_out_v(c.rdx, c.rdy, s, o) : T(0);
            rv[o.kv] = r;
            if (fv && (o.mv & MB_INNER)) fv[o.kv] = r;
            r2 = (double)r * (double)r;
            b2 = (double)b_v * (double)b_v;
        }
        tree256x2(r2, b2, lds);
        if (threadIdx.x == 0) {
            const int q = g.nbxu * g.nbyu + bx + g.nbxv * by;
            Pr[q] = r2;
            if (Pb) Pb[q] = b2;
        }
    }
}

// ===========================================================================
// One iteration of gauss_seidel_smoother! (update_preconditioners.jl:133-150)
// in one launch: the four colour sweeps x[c] += omega (b - A x)[c] / diag[c]
// in the order given, on the u and v points of one tile.  Colours 1
// and 2 are the u points with 1 + mod(i - j, 2) == colour, 3 and 4 the v
// points with 3 + mod(i - j, 2) (get_preconditioner,
// update_preconditioners.jl:7-43).  A point's update reads its neighbours
// within one point, so the tile stages a window with a halo of SM_H = 4
// points; sweep s updates its colour inside the window shrunk by s points,
// whose neighbours hold the values of sweep s - 1, and the fourth sweep
// covers the tile.  Halo points are updated by the neighbouring tiles with
// the same inputs and arithmetic, and only the tile's own points are
// written, into a second buffer (xu_out, xv_out): the other tiles read the
// inputs of the iteration from the first.  Every update has the arithmetic of
// op_u / op_v and of the one-colour sweep, so the result is bit-identical to
// four sweeps of one colour each.
constexpr int SM_H = 4;  // halo points

// A TX x TY tile: window of PX x PY points (the tile and its halo), of which
// the CX x CY cells starting one point in are computed.  Points at
// [py][px] = (i0 - SM_H - 1 + px, j0 - SM_H - 1 + py), px in 1..PX (index 0
// unused); cells and corners with the same origin.  Window position (x, y)
// of a point is px = x + 1, py = y + 1, as optile_u / optile_v expect.
template <int TX, int TY>
struct SmoothShape {
    static constexpr int PX = TX + 2 * SM_H, PY = TY + 2 * SM_H;
    static constexpr int CX = PX - 1, CY = PY - 1;
    static constexpr int SLOTS = (PX * PY + 255) / 256;   // window points per thread
    static constexpr int CSLOTS = (CX * CY + 255) / 256;  // cells per thread
};

template <typename T, int TX, int TY>
struct SmoothWin {
    using S = SmoothShape<TX, TY>;
    T U[S::PY + 1][S::PX + 2];
    T V[S::PY + 1][S::PX + 2];
    T rxx[S::CY + 1][S::CX + 2];
    T ryy[S::CY + 1][S::CX + 2];
    T ext[S::CY + 1][S::CX + 2];
    T rxy[S::CY + 1][S::CX + 2];
};

// The coefficients one window point's update reads.
template <typename T>
struct SmoothPoint {
    PointCoef<T> pc;
    T bu, du, bv, dv;  // right-hand side and diagonal at the u and the v point
};

// Tile shapes of the smoother (the autotuner's candidates): 16 x 16, 32 x 16
// and 16 x 32 points.  Any shape gives the same bits: a point's update does
// not depend on the tile it is computed in.
template <typename T, int TX, int TY>
__global__ void __launch_bounds__(256) k_smooth4(GridDims g, OpCoef<T> c, const T *xu, const T *xv, T *xu_out,
                                                 T *xv_out, const T *bu, const T *bv, const T *du, const T *dv,
                                                 T omega, int order, int ntx, int nty, int nblk, int cols)
{
    using S = SmoothShape<TX, TY>;
    __shared__ SmoothWin<T, TX, TY> s;
    int bx, by;
    if (!xcd_band_tile(ntx, nty, nblk, cols != 0, bx, by)) return;
    const int i0 = bx * TX, j0 = by * TY;
    const int ox = i0 - SM_H, oy = j0 - SM_H;  // window position 0
    // stage the window and load the coefficients the four sweeps read
    SmoothPoint<T> sp[S::SLOTS];
#pragma unroll
    for (int k = 0; k < S::SLOTS; ++k) {
        const int q = threadIdx.x + 256 * k;
        const int x = q % S::PX, y = q / S::PX, i = ox + x, j = oy + y;
        PointCoef<T> &pc = sp[k].pc;
        pc.oku = q < S::PX * S::PY && i >= 0 && j >= 0 && i < g.nxu && j < g.nyu;
        pc.okv = q < S::PX * S::PY && i >= 0 && j >= 0 && i < g.nxv && j < g.nyv;
        pc.ku = i + g.nxu * j;
        pc.kv = i + g.nxv * j;
        pc.ui = pc.um = pc.vi = pc.vm = false;
        pc.bu = pc.hu = pc.bv = pc.hv = T(0);
        sp[k].bu = sp[k].du = sp[k].bv = sp[k].dv = T(0);
        T u = T(0), v = T(0);
        if (pc.oku) {
            u = xu[pc.ku];
            pc.ui = c.ui[pc.ku];
            pc.um = c.um[pc.ku];
            pc.bu = c.bu[pc.ku];
            pc.hu = c.hu[pc.ku];
            sp[k].bu = bu[pc.ku];
            sp[k].du = du[pc.ku];
        }
        if (pc.okv) {
            v = xv[pc.kv];
            pc.vi = c.vi[pc.kv];
            pc.vm = c.vm[pc.kv];
            pc.bv = c.bv[pc.kv];
            pc.hv = c.hv[pc.kv];
            sp[k].bv = bv[pc.kv];
            sp[k].dv = dv[pc.kv];
        }
        if (q < S::PX * S::PY) {
            s.U[y + 1][x + 1] = u;
            s.V[y + 1][x + 1] = v;
        }
    }
    // cell (a, b) = (ox + q % CX, oy + q / CX) at [1 + q / CX][1 + q % CX]
    CellCoef<T> cc[S::CSLOTS];
#pragma unroll
    for (int k = 0; k < S::CSLOTS; ++k) {
        const int q = threadIdx.x + 256 * k;
        cell_prefetch_at(g, c, ox + q % S::CX, oy + q / S::CX, q < S::CX * S::CY, cc[k]);
    }
    for (int sw = 1; sw <= 4; ++sw) {
        const int colour = (order >> (4 * (sw - 1))) & 15;
        __syncthreads();  // the window holds the values after sweep sw - 1
        // sweep sw updates window positions [sw, P - sw), which read the
        // cells at indices [sw, P - sw]
#pragma unroll
        for (int k = 0; k < S::CSLOTS; ++k) {
            const int q = threadIdx.x + 256 * k;
            const int cx = 1 + q % S::CX, cy = 1 + q / S::CX;
            if (q < S::CX * S::CY && cx >= sw && cy >= sw && cx <= S::PX - sw && cy <= S::PY - sw)
                cell_eval(c, cc[k], cx, cy, s);
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < S::SLOTS; ++k) {
            const int q = threadIdx.x + 256 * k;
            const int x = q % S::PX, y = q / S::PX;
            if (q >= S::PX * S::PY || x < sw || y < sw || x >= S::PX - sw || y >= S::PY - sw) continue;
            const PointCoef<T> &pc = sp[k].pc;
            const int i = ox + x, j = oy + y;
            if (colour <= 2) {
                if (pc.oku && pc.ui && ((i - j) & 1) == colour - 1) {
                    const T r = sp[k].bu - optile_u(c, s, pc, x, y);
                    s.U[y + 1][x + 1] = s.U[y + 1][x + 1] + (omega * r) / sp[k].du;
                }
            } else if (pc.okv && pc.vi && ((i - j) & 1) == colour - 3) {
                const T r = sp[k].bv - optile_v(c, s, pc, x, y);
                s.V[y + 1][x + 1] = s.V[y + 1][x + 1] + (omega * r) / sp[k].dv;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < S::SLOTS; ++k) {
        const int q = threadIdx.x + 256 * k;
        const int x = q % S::PX, y = q / S::PX;
        if (q >= S::PX * S::PY || x < SM_H || y < SM_H || x >= SM_H + TX || y >= SM_H + TY) continue;
        if (sp[k].pc.oku) xu_out[sp[k].pc.ku] = s.U[y + 1][x + 1];
        if (sp[k].pc.okv) xv_out[sp[k].pc.kv] = s.V[y + 1][x + 1];
    }
}

// ===========================================================================
// The whole smoothing of a small grid in one workgroup: nsmooth iterations of
// gauss_seidel_smoother! (update_preconditioners.jl:133-150), each the four
// colour sweeps in `order`, with the grid staged in LDS once and block
// barriers between the sweeps, so that a V-cycle's smoothing is one launch
// instead of one per iteration.  The window is the grid with a border of one
// absent point: window position (x, y) is the point (x - 1, y - 1), its value
// at [y + 1][x + 1] and its cell at [y + 1][x + 1] as optile_u / optile_v
// expect.  A point's update is that of k_smooth4 (the arithmetic of op_u /
// op_v and of the one-colour sweep), so the bits are the same.  The result
// goes to xu_out, xv_out, which may be xu, xv: every read of x precedes the
// first barrier and every write follows the last.
// A sweep is a chain of LDS reads, arithmetic and two barriers, once per slot.
// Threads take the grid's points and not the border, which is staged as zero
// once, so the 80 x 10 grid (891 points, 984 cells, 1,079 with the border)
// has one slot: 24.7 -> 22.4 us in FP64, 18.5 -> 17.0 us in FP32.  What remains
// is that chain, about 0.85 us a sweep: the points of one colour in whole
// wavefronts, so that the others skip the update, was slower (23.1, 18.1 us).
constexpr int SMG_THREADS = 1024;
constexpr int SMG_MAX_SLOTS = 2;  // points, and cells, per thread

// Rows of a 2-D array in dynamic LDS.
template <typename T>
struct LdsRows {
    T *p;
    int ld;
    __device__ __forceinline__ T *operator[](int y) const { return p + y * ld; }
};

template <typename T>
struct SmoothGridWin {
    LdsRows<T> U, V, rxx, ryy, ext, rxy;
};

// Extents of the whole-grid window: PX x PY points and CX x CY cells, the
// cell q = (q % CX - 1, q / CX - 1) at [1 + q / CX][1 + q % CX]; U and V have
// PY + 1 rows of PX + 2, the cell arrays CY + 1 rows of CX + 2.
struct SmoothGridDims {
    int PX, PY, CX, CY;
    __host__ __device__ explicit SmoothGridDims(const GridDims &g)
        : PX((g.nxu > g.nxv ? g.nxu : g.nxv) + 2), PY((g.nyu > g.nyv ? g.nyu : g.nyv) + 2), CX(PX - 1), CY(PY - 1)
    {
    }
    __host__ __device__ int points() const { return PX * PY; }
    __host__ __device__ int cells() const { return CX * CY; }
    __host__ __device__ int inner() const { return (PX - 2) * (PY - 2); }  // points without the border
    // LDS elements of the six arrays
    __host__ __device__ size_t elems() const
    {
        return 2 * (size_t)(PY + 1) * (PX + 2) + 4 * (size_t)(CY + 1) * (CX + 2);
    }
};

template <typename T, int SLOTS>
__global__ void __launch_bounds__(SMG_THREADS) k_smooth_grid(GridDims g, OpCoef<T> c, const T *xu, const T *xv,
                                                            T *xu_out, T *xv_out, const T *bu, const T *bv,
                                                            const T *du, const T *dv, T omega, int order, int nsmooth)
{
    extern __shared__ __align__(16) unsigned char smg_lds[];
    const SmoothGridDims d(g);
    const int NX = d.PX - 2, NP = d.inner(), CX = d.CX, CY = d.CY;
    SmoothGridWin<T> s;
    {
        T *p = reinterpret_cast<T *>(smg_lds);
        const int lp = d.PX + 2, lc = CX + 2;
        s.U = {p, lp};
        p += (size_t)(d.PY + 1) * lp;
        s.V = {p, lp};
        p += (size_t)(d.PY + 1) * lp;
        s.rxx = {p, lc};
        p += (size_t)(CY + 1) * lc;
        s.ryy = {p, lc};
        p += (size_t)(CY + 1) * lc;
        s.ext = {p, lc};
        p += (size_t)(CY + 1) * lc;
        s.rxy = {p, lc};
    }
    // stage the grid and load the coefficients every sweep reads
    SmoothPoint<T> sp[SLOTS];
    T u[SLOTS], v[SLOTS];
#pragma unroll
    for (int k = 0; k < SLOTS; ++k) {
        const int q = threadIdx.x + SMG_THREADS * k;
        const int i = q % NX, j = q / NX;
        PointCoef<T> &pc = sp[k].pc;
        pc.oku = q < NP && i < g.nxu && j < g.nyu;
        pc.okv = q < NP && i < g.nxv && j < g.nyv;
        pc.ku = i + g.nxu * j;
        pc.kv = i + g.nxv * j;
        pc.ui = pc.um = pc.vi = pc.vm = false;
        pc.bu = pc.hu = pc.bv = pc.hv = T(0);
        sp[k].bu = sp[k].du = sp[k].bv = sp[k].dv = T(0);
        u[k] = v[k] = T(0);
        if (pc.oku) {
            u[k] = xu[pc.ku];
            pc.ui = c.ui[pc.ku];
            pc.um = c.um[pc.ku];
            pc.bu = c.bu[pc.ku];
            pc.hu = c.hu[pc.ku];
            sp[k].bu = bu[pc.ku];
            sp[k].du = du[pc.ku];
        }
        if (pc.okv) {
            v[k] = xv[pc.kv];
            pc.vi = c.vi[pc.kv];
            pc.vm = c.vm[pc.kv];
            pc.bv = c.bv[pc.kv];
            pc.hv = c.hv[pc.kv];
            sp[k].bv = bv[pc.kv];
            sp[k].dv = dv[pc.kv];
        }
    }
    CellCoef<T> cc[SLOTS];
#pragma unroll
    for (int k = 0; k < SLOTS; ++k) {
        const int q = threadIdx.x + SMG_THREADS * k;
        cell_prefetch_at(g, c, q % CX - 1, q / CX - 1, q < CX * CY, cc[k]);
    }
    // the border, then the points
    for (int q = threadIdx.x; q < 2 * (d.PY + 1) * (d.PX + 2); q += SMG_THREADS) s.U.p[q] = T(0);  // U, then V
    __syncthreads();
#pragma unroll
    for (int k = 0; k < SLOTS; ++k) {
        const int q = threadIdx.x + SMG_THREADS * k;
        if (q >= NP) continue;
        const int x = 1 + q % NX, y = 1 + q / NX;
        s.U[y + 1][x + 1] = u[k];
        s.V[y + 1][x + 1] = v[k];
    }
    for (int it = 0; it < nsmooth; ++it) {
        for (int sw = 0; sw < 4; ++sw) {
            const int colour = (order >> (4 * sw)) & 15;
            __syncthreads();  // the window holds the values after the previous sweep
#pragma unroll
            for (int k = 0; k < SLOTS; ++k) {
                const int q = threadIdx.x + SMG_THREADS * k;
                if (q < CX * CY) cell_eval(c, cc[k], 1 + q % CX, 1 + q / CX, s);
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < SLOTS; ++k) {
                const int q = threadIdx.x + SMG_THREADS * k;
                if (q >= NP) continue;
                const int i = q % NX, j = q / NX, x = i + 1, y = j + 1;
                const PointCoef<T> &pc = sp[k].pc;
                if (colour <= 2) {
                    if (pc.oku && pc.ui && ((i - j) & 1) == colour - 1) {
                        const T r = sp[k].bu - optile_u(c, s, pc, x, y);
                        s.U[y + 1][x + 1] = s.U[y + 1][x + 1] + (omega * r) / sp[k].du;
                    }
                } else if (pc.okv && pc.vi && ((i - j) & 1) == colour - 3) {
                    const T r = sp[k].bv - optile_v(c, s, pc, x, y);
                    s.V[y + 1][x + 1] = s.V[y + 1][x + 1] + (omega * r) / sp[k].dv;
                }
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < SLOTS; ++k) {
        const int q = threadIdx.x + SMG_THREADS * k;
        if (q >= NP) continue;
        const int x = 1 + q % NX, y = 1 + q / NX;
        if (sp[k].pc.oku) xu_out[sp[k].pc.ku] = s.U[y + 1][x + 1];
        if (sp[k].pc.okv) xv_out[sp[k].pc.kv] = s.V[y + 1][x + 1];
    }
}

// ===========================================================================
// Restricted additive Schwarz (SharedMemorySpec, src/SharedMemorySpec.jl):
// moving velocities between the full grid and a subdomain context on the
// same device.  A subdomain covers the cells [i0, i0 + nxg) x [j0, j0 + nyg)
// of the full grid (its u points i0 .. i0 + nxg, its v points j0 .. j0 + nyg).
struct RasPart {
    int i0, j0, nxg, nyg;
    int leave_i1, leave_im, leave_j1, leave_jn;  // edges where the partition of unity stays 1
    int overlap;
};

// schwarzRestrictVelocities! (SharedMemorySpec.jl:306-331): the subdomain's
// u and v are the full model's on its points (blockIdx.y 0: u, 1: v).
__global__ void k_ras_restrict(RasPart p, int nxuf, int nxvf, const double *Uf, const double *Vf, double *Ug,
                               double *Vg)
{
    const bool v = blockIdx.y != 0;
    const int mx = v ? p.nxg : p.nxg + 1, my = v ? p.nyg + 1 : p.nyg;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= mx * my) return;
    const int i = k % mx, j = k / mx;
    if (v)
        Vg[k] = Vf[(p.i0 + i) + nxvf * (p.j0 + j)];
    else
        Ug[k] = Uf[(p.i0 + i) + nxuf * (p.j0 + j)];
}

// One factor of schwarzPartitionOfUnity (SharedMemorySpec.jl:395-407) at the
// 1-based index i of m: min(1, (i - 1) / ov, (m - i) / ov), an edge left out
// where it is kept at 1.
__device__ __forceinline__ double ras_pou(int i, int m, bool leave_lo, bool leave_hi, int ov)
{
    const double lo = leave_lo ? INFINITY : (double)(i - 1) / (double)ov;
    const double hi = leave_hi ? INFINITY : (double)(m - i) / (double)ov;
    return fmin(1.0, fmin(lo, hi));
}

// schwarzProlongVelocities! (SharedMemorySpec.jl:351-382) for one
// subdomain: u += ((1 - damping) pou) u_g on its points, with the partition
// of unity ramping over 2 overlap points across u's x edges and 2 overlap - 1
// across its y edges (the other way round for v).
__global__ void k_ras_prolong(RasPart p, int nxuf, int nxvf, double *Uf, double *Vf, const double *Ug,
                              const double *Vg, double one_minus_damping)
{
    const bool v = blockIdx.y != 0;
    const int mx = v ? p.nxg : p.nxg + 1, my = v ? p.nyg + 1 : p.nyg;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= mx * my) return;
    const int i = k % mx, j = k / mx;
    const int ovx = v ? 2 * p.overlap - 1 : 2 * p.overlap, ovy = v ? 2 * p.overlap : 2 * p.overlap - 1;
    const double pou = ras_pou(i + 1, mx, p.leave_i1, p.leave_im, ovx) * ras_pou(j + 1, my, p.leave_j1, p.leave_jn, ovy);
    const double t = one_minus_damping * pou;
    if (v) {
        double *a = &Vf[(p.i0 + i) + nxvf * (p.j0 + j)];
        *a = *a + t * Vg[k];
    } else {
        double *a = &Uf[(p.i0 + i) + nxuf * (p.j0 + j)];
        *a = *a + t * Ug[k];
    }
}

// A subdomain model as schwarzModel builds it (SharedMemorySpec.jl:181-287)
// from the full model's fields, with the initial fields of setup_fields
// (src/Fields/Fields.jl:26-115): bed, thickness, grounded fraction, u, v,
// viscosity, glen_b and the Weertman coefficient and accumulation arrays
// sliced from the full grid; eta_av the bottom viscosity level; quad_f2 =
// h / (3 eta_av) on the mask; dsdh and the u/v grounded fractions 1; the
// wavelet masks all set; every other field 0.  One thread per entry of the
// largest of the subdomain's h, u, v and sigma grids.
struct RasRefresh {
    RasPart p;
    int nxf, nyf, ns;  // full h grid, sigma levels
    const double *b, *h, *gf, *wc, *acc, *u, *v, *eta, *glenb;  // full-grid sources
    double *f[WAVI_NFIELDS];                                   // subdomain fields (nullptr: not a double field)
    uint8_t *mwu, *mwv;
    const uint8_t *hm;                                         // subdomain h mask
};

__global__ void k_ras_refresh(RasRefresh r)
{
    const RasPart &p = r.p;
    const int nxg = p.nxg, nyg = p.nyg, nh = nxg * nyg;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < nh) {
        const int i = k % nxg, j = k / nxg;
        const int sidx = (p.i0 + i) + r.nxf * (p.j0 + j);
        for (int id = WAVI_H_B; id <= WAVI_P_ACCUMULATION_RATE; ++id) r.f[id][k] = 0.0;
        r.f[WAVI_H_B][k] = r.b[sidx];
        r.f[WAVI_H_H][k] = r.h[sidx];
        r.f[WAVI_H_GROUNDED_FRACTION][k] = r.gf[sidx];
        r.f[WAVI_P_WEERTMAN_C][k] = r.wc[sidx];
        r.f[WAVI_P_ACCUMULATION_RATE][k] = r.acc[sidx];
        r.f[WAVI_H_DSDH][k] = 1.0;
        const double eta0 = r.eta[sidx];
        r.f[WAVI_H_ETA_AV][k] = eta0;
        r.f[WAVI_H_QUAD_F2][k] = r.hm[k] ? r.h[sidx] / (3.0 * eta0) : 0.0;
    }
    const int nu = (nxg + 1) * nyg;
    if (k < nu) {
        const int i = k % (nxg + 1), j = k / (nxg + 1);
        for (int id = WAVI_U_S; id <= WAVI_U_RESIDUAL; ++id) r.f[id][k] = 0.0;
        r.f[WAVI_U_U][k] = r.u[(p.i0 + i) + (r.nxf + 1) * (p.j0 + j)];
        r.f[WAVI_U_GROUNDED_FRACTION][k] = 1.0;
        r.f[WAVI_WU_WAVELETS][k] = 0.0;
        r.f[WAVI_WU_CORRECTION_COARSE][k] = 0.0;
        r.mwu[k] = 1;
    }
    const int nv = nxg * (nyg + 1);
    if (k < nv) {
        const int i = k % nxg, j = k / nxg;
        for (int id = WAVI_V_S; id <= WAVI_V_RESIDUAL; ++id) r.f[id][k] = 0.0;
        r.f[WAVI_V_V][k] = r.v[(p.i0 + i) + r.nxf * (p.j0 + j)];
        r.f[WAVI_V_GROUNDED_FRACTION][k] = 1.0;
        r.f[WAVI_WV_WAVELETS][k] = 0.0;
        r.f[WAVI_WV_CORRECTION_COARSE][k] = 0.0;
        r.mwv[k] = 1;
    }
    if (k < nh * r.ns) {
        const int l = k / nh, q = k % nh;
        const int i = q % nxg, j = q / nxg;
        const int sidx = (p.i0 + i) + r.nxf * ((p.j0 + j) + r.nyf * l);
        r.f[WAVI_S_ETA][k] = r.eta[sidx];
        r.f[WAVI_S_GLEN_B][k] = r.glenb[sidx];
    }
}

// u = damping u, v = damping v on the full grid (SharedMemorySpec.jl:134-135).
__global__ void k_scale_uv(double *u, int nu, double *v, int nv, double a)
{
    const bool isv = blockIdx.y != 0;
    double *x = isv ? v : u;
    const int n = isv ? nv : nu;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) x[k] = a * x[k];
}

// ===========================================================================
// Coarse CG: IterativeSolvers.cg! on A_c = R A P (update_preconditioners.jl:73)
// with x0 the cached warm start: two kernels per iteration (one per global
// sum) and no host round trip.  Kernels that end in a reduction write one partial per 16x16
// block; the next kernel folds them with the canonical tree in every
// workgroup (all get the same bits), so no workgroup waits for another inside
// a kernel.  Scalars a kernel publishes are double-buffered by iteration
// parity and every workgroup writes the same value; a kernel never reads a
// scalar that another workgroup of the same kernel writes.
// PRE = true (inside the flexible CG's linear solves only) runs
// preconditioned CG with M = D^-1, D = |diag A_c| (k_coarse_diag): the
// direction takes D^-1 r, alpha and beta take (r, D^-1 r), and the stop test
// stays on ||r||.  PRE = false is cg! as the reference runs it.

// Stop report of a coarse CG in host-mapped pinned memory: written once, by
// the launch that stops, so the host learns of the stop without a copy on
// the stream.
struct CGMHostFlag {
    int done;
    int iters;
    int gave_up;  // the resident CG did, and k_cg_solve1 ran in its place
};

struct CGScalars {
    double res[2];    // residual norm by iteration parity (written by k_cg_step)
    double tol;       // max(reltol ||r0||, abstol)
    double alpha;     // step length whose x += alpha u is still to be applied (written by k_cg_update)
    int it[2];        // iterations done, by parity
    int done;         // sticky stop flag, written only by k_cg_step
    int iters;        // iterations at termination
    double rz[2];     // Jacobi-preconditioned CG: (r, D^-1 r) by parity (written by k_cg_step)
    int abort;        // a workgroup of k_cg_resident gave up waiting
};

// The FP64 coarse CG works in an arena of zero-padded 2-D arrays shared by
// the u grid, the v grid and the h cells: point (i, j) at (i + 16) + px (j +
// 16), px = 16 (nbx + 1), with a border of one tile that stays zero (the next
// row's left border is a row's right one).  A tile's
// rows are then aligned, u and v of a point come in one 16-byte load, every
// window, halo and store is unconditional at a 32-bit offset from a uniform
// base, and what a tile stores past the end of a grid is zero.  Guarded
// loads from the compact arrays at clamped indices took about half of the
// VALU instructions of an iteration.  k_cg_setup fills it.
enum CGPair {        // (u, v) pairs, ns each
    CG_R = 0,        // residual r
    CG_P = 1,        // search direction u, by iteration parity (two arrays)
    CG_X = 3,        // solution
    CG_Q = 4,        // c = A_c u
    CG_H = 5,        // thickness on u and v points, 0 off the masks
    CG_B = 6,        // beta_eff on u and v points, 0 off the masks
    CG_CELL = 7,     // per h cell: (h*eta_av, dimp)
    CG_DINV = 8,     // Jacobi: 1 / |diag(A_c)|, 0 off the wavelet masks
    CG_NPAIR = 9
};
enum { CB_INNER_U = 1, CB_INNER_V = 2, CB_WAVELET_U = 4, CB_WAVELET_V = 8 };  // mask bits of a point

struct CGLayout {
    double2 *F;       // pair array A at F + A * ns, then the corners' h*eta_av (ns doubles)
    uint8_t *M;       // mask bits (CB_*)
    unsigned px, ns;  // row pitch, array stride
    __device__ __forceinline__ unsigned at(int i, int j) const
    {
        return (unsigned)(i + TILE) + __umul24(px, (unsigned)(j + TILE));
    }
    // (dx, dy) from index k, dy >= -TILE: the product of what is not negative
    // (a signed 24-bit one would end at a pitch of 2^23, half of the largest)
    __device__ __forceinline__ unsigned from(unsigned k, int dx, int dy) const
    {
        return (k - (unsigned)TILE * px) + (unsigned)dx + __umul24(px, (unsigned)(dy + TILE));
    }
    __device__ __forceinline__ double2 *pair(int a) const { return F + (size_t)a * ns; }
    __device__ __forceinline__ double *corner() const { return reinterpret_cast<double *>(F + (size_t)CG_NPAIR * ns); }
};

// Element k of an array, addressed by a 32-bit byte offset from its uniform
// base (the scalar-base form of the global loads and stores).  BIG: of an
// array of 4 GiB and more, by a 64-bit address of each lane's own.
template <bool BIG, typename V>
__device__ __forceinline__ V &elem(V *p, unsigned k)
{
    if constexpr (BIG) return p[k];
    typedef typename std::conditional<std::is_const<V>::value, const char, char>::type C;
    return *reinterpret_cast<V *>(reinterpret_cast<C *>(p) + (size_t)(unsigned)(k * (unsigned)sizeof(V)));
}

template <typename V>
__device__ __forceinline__ V &elem32(V *p, unsigned k)
{
    return elem<false>(p, k);
}

struct CGArgs {
    GridDims g;
    CGLayout Lo;
    double rdx, rdy;
    double *Pr, *Pd, *Pb;
    double *Pz;                       // Jacobi: partials of (r, D^-1 r)
    CGScalars *st;
    CGMHostFlag *hflag;   // host-mapped stop report
    double tol_coarse, reltol;
    int maxiter;
    int nblk;         // launched workgroups, a multiple of 8
};

// What the set-up and the end of the CG read and write besides: the compact
// arrays.
struct CGIo {
    OpCoef<double> c;
    int levels;
    const uint8_t *mwu, *mwv;
    const double *bu, *bv;            // right-hand side
    double *xu, *xv;                  // warm start in, solution out
    const double *tu, *tv;            // P x0
    const double *dinvu, *dinvv;      // Jacobi: 1 / |diag(A_c)|, 0 off the wavelet masks
    double *eu, *ev;                  // the V-cycle's correction, += P x
    const int *abort;                 // CGScalars::abort
    int resident;                     // the CG ran as k_cg_resident
};

// XCD-aware tile order: workgroups are dispatched round-robin over the 8
// XCDs, so workgroup w takes tile (w % 8) * (nblk / 8) + w / 8 and each XCD
// walks one contiguous band of tiles in row-major order (whole grid rows of
// the arrays, which the coarse-CG kernels read fastest: a column-major walk
// was measured 4.5% slower for k_cgm_iter at 1280 x 160).
__device__ __forceinline__ int xcd_tile(int nblk)
{
    const int w = blockIdx.x;
    return (w & 7) * (nblk >> 3) + (w >> 3);
}

__device__ __forceinline__ int band_tile(const GridDims &g, int L, int &bx, int &by)
{
    bx = L % g.nbx;
    by = L / g.nbx;
    return L;
}

// setup (t = P x0 computed beforehand): r = b - R A t, x = x0, u = 0, the
// coefficients and mask bits into the arena, partials of ||r0||^2 and ||b||^2
// (PRE: also of (r0, D^-1 r0)); resets the scalars.
template <bool PRE, bool BIG>
__global__ void __launch_bounds__(256) k_cg_setup(CGArgs a, CGIo io)
{
    __shared__ OpLds<double> s;
    __shared__ double lds[8];
    const GridDims &g = a.g;
    const int L = xcd_tile(a.nblk);
    if (L >= g.nbx * g.nby) return;
    if (L == 0 && threadIdx.x == 0) {
        a.st->done = 0;
        a.st->iters = 0;
        a.st->it[0] = 0;
        a.st->it[1] = 0;
        a.st->alpha = 0.0;
        a.st->abort = 0;
        // also reset on the stream: launches queued past the previous
        // CG's stop, which rewrite the report, may still have been running
        // when the host reset it
        a.hflag->done = 0;
        a.hflag->iters = 0;
        a.hflag->gave_up = 0;
    }
    int bx, by;
    band_tile(g, L, bx, by);
    const bool has_u = bx < g.nbxu && by < g.nbyu, has_v = bx < g.nbxv && by < g.nbyv;
    const int i0 = bx * TILE, j0 = by * TILE;
    const int lx = threadIdx.x & 15, ly = threadIdx.x >> 4;
    OpOwn<double> o;
    op_own_index(g, i0 + lx, j0 + ly, o.oku, o.okv, o.ku, o.kv);
    const double bu = ld_or(o.oku, io.bu, o.ku, 0.0), bv = ld_or(o.okv, io.bv, o.kv, 0.0);
    const double xu = ld_or(o.oku, io.xu, o.ku, 0.0), xv = ld_or(o.okv, io.xv, o.kv, 0.0);
    const double zu = PRE ? ld_or(o.oku, io.dinvu, o.ku, 0.0) : 0.0, zv = PRE ? ld_or(o.okv, io.dinvv, o.kv, 0.0) : 0.0;
    const OpCoef<double> &c = io.c;
    op_restrict_tile(g, c, MaskSep<true>{c.ui, c.um, c.vi, c.vm, io.mwu, io.mwv}, io.levels, io.tu, io.tv, i0, j0, s, o);
    const double ru = (o.mu & MB_WAVELET) ? bu - s.h.t[0][ly][lx] : bu, rv = (o.mv & MB_WAVELET) ? bv - s.h.t[1][ly][lx] : bv;
    const unsigned at = a.Lo.at(i0 + lx, j0 + ly);
    elem<BIG>(a.Lo.pair(CG_R), at) = make_double2(ru, rv);
    elem<BIG>(a.Lo.pair(CG_P), at) = make_double2(0.0, 0.0);
    elem<BIG>(a.Lo.pair(CG_X), at) = make_double2(xu, xv);
    elem<BIG>(a.Lo.pair(CG_H), at) = make_double2(o.hu, o.hv);
    elem<BIG>(a.Lo.pair(CG_B), at) = make_double2(o.bu, o.bv);
    elem<BIG>(a.Lo.pair(CG_CELL), at) = make_double2(o.heta, o.dimp);
    if constexpr (PRE) elem<BIG>(a.Lo.pair(CG_DINV), at) = make_double2(zu, zv);
    elem<BIG>(a.Lo.corner(), at) = o.hetac;
    elem<BIG>(a.Lo.M, at) = (uint8_t)(((o.mu & MB_INNER) ? CB_INNER_U : 0) | ((o.mv & MB_INNER) ? CB_INNER_V : 0) |
                           ((o.mu & MB_WAVELET) ? CB_WAVELET_U : 0) | ((o.mv & MB_WAVELET) ? CB_WAVELET_V : 0));
    double r2u = ru * ru, r2v = rv * rv, b2u = bu * bu, b2v = bv * bv;
    tree256x2(r2u, r2v, lds);
    tree256x2(b2u, b2v, lds);
    double z2u = 0.0, z2v = 0.0;
    if constexpr (PRE) {
        z2u = ru * (zu * ru);
        z2v = rv * (zv * rv);
        tree256x2(z2u, z2v, lds);
    }
    if (threadIdx.x == 0) {
        if (has_u) {
            a.Pr[bx + g.nbxu * by] = r2u;
            a.Pb[bx + g.nbxu * by] = b2u;
            if constexpr (PRE) a.Pz[bx + g.nbxu * by] = z2u;
        }
        if (has_v) {
            const int q = g.nbxu * g.nbyu + bx + g.nbxv * by;
            a.Pr[q] = r2v;
            a.Pb[q] = b2v;
            if constexpr (PRE) a.Pz[q] = z2v;
        }
    }
}

// The end of a CG on one tile: (x, y) = the solution at the thread's point,
// back into the compact warm start, and e += P x at the inner points.
template <typename T>
__device__ __forceinline__ void cg_finish_tile(const GridDims &g, int levels, int bx, int by, T x, T y, unsigned mb,
                                               T *xu, T *xv, T *eu, T *ev)
{
    __shared__ TilePair<T> t, m;
    const int lx = threadIdx.x & 15, ly = threadIdx.x >> 4;
    bool oku, okv;
    int ku, kv;
    op_own_index(g, bx * TILE + lx, by * TILE + ly, oku, okv, ku, kv);
    const T e_u = ld_or(oku, (const T *)eu, ku, T(0)), e_v = ld_or(okv, (const T *)ev, kv, T(0));
    if (oku) xu[ku] = x;
    if (okv) xv[kv] = y;
    t[0][ly][lx] = (mb & CB_WAVELET_U) ? x : T(0);
    t[1][ly][lx] = (mb & CB_WAVELET_V) ? y : T(0);
    __syncthreads();
    haar_pair<false, T>(levels, t, m);
    if (mb & CB_INNER_U) eu[ku] = e_u + t[0][ly][lx];
    if (mb & CB_INNER_V) ev[kv] = e_v + t[1][ly][lx];
}

template <bool BIG>
__global__ void __launch_bounds__(256) k_cg_finish(CGArgs a, CGIo io)
{
    const int L = xcd_tile(a.nblk);
    if (L >= a.g.nbx * a.g.nby) return;
    int bx, by;
    band_tile(a.g, L, bx, by);
    const unsigned at = a.Lo.at(bx * TILE + (int)(threadIdx.x & 15), by * TILE + (int)(threadIdx.x >> 4));
    const bool resident = io.resident && *io.abort == 0;  // the resident CG leaves x in CG_Q
    const double2 x = elem<BIG>(a.Lo.pair(resident ? CG_Q : CG_X), at);
    cg_finish_tile<double>(a.g, io.levels, bx, by, x.x, x.y, elem<BIG>(a.Lo.M, at), io.xu, io.xv, io.eu, io.ev);
}

// A CG scalar written by an earlier kernel, read as a vector load: a scalar
// load of it comes back under the same wait as the kernel's arguments, which
// the launch's later vector loads (the partials) need first, so its round
// trip would come before theirs.  The index is a zero the compiler cannot
// see through (a register move, not a load), which makes the load a vector
// load, waited for where its value is used.
template <typename V>
__device__ __forceinline__ V cg_scalar(const V *p)
{
    int z;
    asm volatile("v_mov_b32 %0, 0" : "=v"(z));
    return p[z];
}

// Offset of the k-th coarse row (or column) that the point next to a tile
// takes from the neighbour, relative to the tile's first: before the tile
// the neighbour's last point 15, whose row of P has the terms 16 - B, .., 8,
// 12, 14, 15 (all +1), after it the neighbour's first point 0 with the terms
// 0, 1, 2, 4, 8 (+1, then all -1).  N = LEV + 2 of them, in increasing order.
template <int LEV>
__device__ __forceinline__ int haar_halo_offset(bool after, int k)
{
    return after ? 16 + ((1 << k) >> 1) : -((2 << LEV) >> k);
}

// A row of P on the terms at v + off[0..N): + for the first `plus` details,
// then -.
template <int LEV, typename T>
struct HaarRow {
    T x[LEV + 2];
    __device__ __forceinline__ void load(const T *v, const int (&off)[LEV + 2])
    {
#pragma unroll
        for (int k = 0; k < LEV + 2; ++k) x[k] = v[off[k]];
    }
    __device__ __forceinline__ T sum(int plus) const
    {
        T a = x[0];
#pragma unroll
        for (int k = 0; k <= LEV; ++k) a = add_sign(a, x[k + 1], k >= plus);
        return a;
    }
};

// The terms of haar_halo_offset (stride st): the last point of a block (all +)
// or its first (all -).
template <int LEV>
__device__ __forceinline__ void haar_halo_terms(int st, int (&off)[LEV + 2])
{
#pragma unroll
    for (int k = 0; k < LEV + 2; ++k) off[k] = k * st;
}

// The terms of row i of a 16-point line in increasing column order: the
// block's first, the e_h of i's set bits (h descending), then of its clear
// bits (h ascending).  Returns the number of set bits.
template <int LEV>
__device__ __forceinline__ int haar_row_terms(int i, int (&off)[LEV + 2])
{
    off[0] = i & ~((2 << LEV) - 1);
    int plus = 0;
#pragma unroll
    for (int h = 0; h <= LEV; ++h) plus += (i >> h) & 1;
    int up = 0;
#pragma unroll
    for (int k = 1; k < LEV + 2; ++k) off[k] = 0;
#pragma unroll
    for (int h = LEV; h >= 0; --h) {  // slot of e_h: set bits count down from h = LEV, clear bits come last in reverse
        const bool set = (i >> h) & 1;
        const int e = (i & ~((2 << h) - 1)) + (1 << h);
        const int clear_below = h - (plus - up - (set ? 1 : 0));  // clear bits under h
        const int slot = 1 + (set ? up : plus + clear_below);
#pragma unroll
        for (int k = 1; k < LEV + 2; ++k) off[k] = slot == k ? e : off[k];
        up += set ? 1 : 0;
    }
    return plus;
}

// The geometry and the coefficients of a thread's part of a tile, and the
// tile's c = R A P u from its own direction and the coarse halo's.
template <int LEV, bool BIG = false>
struct CgTile {
    using T = double;
    static constexpr int N = LEV + 2;
    int l, w, lx, ly;
    unsigned at0, at, h0, h1;         // arena index of the tile, the own point, the two coarse halo points
    bool rows, after, corner;
    int cx, cy;                       // corner entry
    HaloPos h;
    OpOwn<T> o;
    OpCoefRegs<T> cr;
    unsigned mb, hmb;                 // mask bits of the own and the halo point
    int hoff[N], hplus;               // the halo point's terms in the x pass (wavefronts 2, 3)

    __device__ __forceinline__ void place(const CGLayout &Lo, int i0, int j0)
    {
        lx = threadIdx.x & 15;
        ly = threadIdx.x >> 4;
        l = threadIdx.x & 63;
        w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        at0 = Lo.at(i0, j0);
        at = at0 + lx + __umul24(Lo.px, (unsigned)ly);
    }
    // (apart, so that the first loads do not wait for its arithmetic)
    __device__ __forceinline__ void place_halo(const CGLayout &Lo)
    {
        // the coarse halo, one side per wavefront (left, right, below, above):
        // line k = l / 16 of N, point l % 16 along it; the fifth line and the
        // corner blocks (u below right, v above left) in a second round
        rows = w >= 2;
        after = (w & 1) != 0;
        int di, dj;
        {
            const int c = haar_halo_offset<LEV>(after, l >> 4), q = l & 15;
            di = rows ? q : c;
            dj = rows ? c : q;
        }
        h0 = Lo.from(at0, di, dj);
        const int e = l - 16;  // corner entry of lanes 16..40 of wavefronts 0 (v) and 1 (u)
        cx = e % 5;
        cy = e / 5;
        corner = w < 2 && e >= 0 && e < 25;
        {
            const int c = haar_halo_offset<LEV>(after, 4), q = l & 15;
            di = corner ? haar_halo_offset<LEV>(after, cx) : (rows ? q : c);
            dj = corner ? haar_halo_offset<LEV>(!after, cy) : (rows ? c : q);
        }
        h1 = Lo.from(at0, di, dj);
    }
    // the coefficients, in the order of their first use
    __device__ __forceinline__ void load_coef(const CGLayout &Lo)
    {
        // halo points: wavefront 3 the sides' u, wavefront 2 their v, wavefront 1
        // the corners (u lane 0, v lane 1)
        h = HaloPos{17, 0, 0, 17, w == 3 || (w == 1 && l == 0), w == 2 || (w == 1 && l == 1)};
        if (w >= 2) {
            halo_side(l, h.ux, h.uy);
            h.vx = h.ux;
            h.vy = h.uy;
        }
        cr.hhu = cr.hhv = 0.0;
        const double2 oh = elem<BIG>(Lo.pair(CG_H), at);
        hmb = 0;
        if (w >= 1) {
            const int hx = h.hu ? h.ux : h.vx, hy = h.hu ? h.uy : h.vy;
            const unsigned ha = Lo.from(at0, hx - 1, hy - 1);
            cr.hhu = cr.hhv = elem<BIG>(reinterpret_cast<const double *>(Lo.pair(CG_H)), 2 * ha + (h.hu ? 0 : 1));
            hmb = elem<BIG>(Lo.M, ha);
        }
        const double2 cell = elem<BIG>(Lo.pair(CG_CELL), at);
        o.hetac = elem<BIG>(Lo.corner(), at);
        op_extra_cell(l, cr);
        if (w == 0) {
            const unsigned ea = Lo.from(at0, cr.ex - 1, cr.ey - 1);
            const double2 ce = elem<BIG>(Lo.pair(CG_CELL), ea);
            cr.ec = elem<BIG>(Lo.corner(), ea);
            cr.eh = ce.x;
            cr.ed = ce.y;
        }
        const double2 ob = elem<BIG>(Lo.pair(CG_B), at);
        o.hu = oh.x;
        o.hv = oh.y;
        o.bu = ob.x;
        o.bv = ob.y;
        o.heta = cell.x;
        o.dimp = cell.y;
        if (l < 32) {
            haar_halo_terms<LEV>(17, hoff);
            hplus = l < 16 ? LEV + 1 : 0;
        } else {
            hplus = haar_row_terms<LEV>(l & 15, hoff);
        }
    }
    // un: the direction at the own point; n0, n1: at the coarse halo points.
    // Six barriers; the first is followed by the rest only if go() holds.
    template <class Go>
    __device__ __forceinline__ bool apply(T rdx, T rdy, double2 un, double2 n0, double2 n1, OpLds<T> &s, double2 &c,
                                          Go go)
    {
        s.p.t[0][ly][lx] = un.x;
        s.p.t[1][ly][lx] = un.y;
        {
            const int k = (w & 1) * 5 + (l >> 4), q = l & 15;
            if (rows) {
                s.n.y[0][k][q] = n0.x;
                s.n.y[1][k][q] = n0.y;
                if (l < 16) {
                    s.n.y[0][k + 4][q] = n1.x;
                    s.n.y[1][k + 4][q] = n1.y;
                }
            } else {
                s.n.x[0][k][q] = n0.x;
                s.n.x[1][k][q] = n0.y;
                if (l < 16) {
                    s.n.x[0][k + 4][q] = n1.x;
                    s.n.x[1][k + 4][q] = n1.y;
                } else if (corner) {
                    s.n.c[1 - w][cy][cx] = w == 1 ? n1.x : n1.y;
                }
            }
        }
        __syncthreads();
        if (!go()) return false;
        // y pass: the tile's lines; the columns' lines (40 half lines; lanes
        // 40..63 repeat the first); rows -1 and 16 of the neighbours below and
        // above (lanes 0..15) and the corners (16..20 of wavefronts 0, 1).  The
        // operands of all three are read before the first is used.
        {
            const int q = l & 15, comp = (l >> 4) & 1, half = l >> 5;
            const int hl = l < 40 ? l : l - 40, line = hl < 20 ? hl : hl - 20, lh = hl < 20 ? 0 : 1;
            const int cp = w & 1, side = w >> 1;
            const bool edge = l < 16;
            const T *se = edge ? &s.n.y[cp][5 * side][l] : &s.n.c[cp][0][l < 20 ? l - 16 : 4];
            int off[N];
            haar_halo_terms<LEV>(edge ? 16 : 5, off);
            HaarLineP<LEV, T> own, hal;
            HaarRow<LEV, T> row;
            own.load(&s.p.t[comp][0][q], TILE + 1, half, w);
            hal.load(&s.n.x[0][0][0] + 17 * line, 1, lh, w);
            row.load(se, off);
            own.rows(&s.p.m[comp][0][q], TILE + 1, half, w);
            hal.rows(&s.n.lx[0][0][0] + 17 * line, 1, lh, w);
            const T y = row.sum((edge ? side != 0 : w == 1) ? 0 : LEV + 1);
            if (edge)
                s.n.ly[cp][side][l] = y;
            else if (w < 2 && l < 21)
                s.n.lc[w][l - 16] = y;
        }
        __syncthreads();
        // x pass: the tile's lines and the halo points
        T hu = 0.0, hv = 0.0;
        {
            const int q = l & 15, comp = (l >> 4) & 1, half = l >> 5;
            HaarLineP<LEV, T> own;
            own.load(&s.p.m[comp][q][0], 1, half, w);
            if (w >= 2) {
                const int cp = w == 3 ? 0 : 1, side = (l >> 4) & 1;
                HaarRow<LEV, T> row;
                row.load(l < 32 ? &s.n.lx[cp][5 * side][q] : &s.n.ly[cp][side][0], hoff);
                own.rows(&s.p.t[comp][q][0], 1, half, w);
                const T y = row.sum(hplus);
                hu = hv = (hmb & (w == 3 ? CB_INNER_U : CB_INNER_V)) ? y : 0.0;
            } else {
                int off[N];
                haar_halo_terms<LEV>(1, off);
                HaarRow<LEV, T> row;
                row.load(&s.n.lc[l == 0 ? 0 : 1][0], off);
                own.rows(&s.p.t[comp][q][0], 1, half, w);
                const T y = row.sum(l == 0 ? 0 : LEV + 1);
                hu = hv = (hmb & (l == 0 ? CB_INNER_U : CB_INNER_V)) ? y : 0.0;  // staged by wavefront 1's lanes 0, 1
            }
        }
        __syncthreads();
        o.u = (mb & CB_INNER_U) ? s.p.t[0][ly][lx] : 0.0;
        o.v = (mb & CB_INNER_V) ? s.p.t[1][ly][lx] : 0.0;
        op_cells<false>(rdx, rdy, h, hu, hv, o, cr, s);
        s.h.t[0][ly][lx] = (mb & CB_INNER_U) ? op_out_u(rdx, rdy, s, o) : 0.0;
        s.h.t[1][ly][lx] = (mb & CB_INNER_V) ? op_out_v(rdx, rdy, s, o) : 0.0;
        __syncthreads();
        haar_pair_lev<true, LEV, T>(s.h.t, s.h.m);
        c = make_double2((mb & CB_WAVELET_U) ? s.h.t[0][ly][lx] : 0.0, (mb & CB_WAVELET_V) ? s.h.t[1][ly][lx] : 0.0);
        return true;
    }
};

// beta of iteration it, and the direction z + beta u (z = r, or D^-1 r)
template <bool PRE>
__device__ __forceinline__ double cg_beta(int it, double res, double prev_res, double rz, double prev_rz)
{
    if constexpr (PRE) {
        return it == 0 ? 0.0 : rz / prev_rz;
    } else {
        const double prev = it == 0 ? 1.0 : prev_res;
        return (res * res) / (prev * prev);
    }
}

template <bool PRE>
__device__ __forceinline__ double2 cg_direction(double beta, double2 r, double2 p, double2 dz)
{
    if constexpr (PRE)
        return make_double2(dz.x * r.x + beta * p.x, dz.y * r.y + beta * p.y);
    else
        return make_double2(r.x + beta * p.x, r.y + beta * p.y);
}

// part 1 (iteration parity par): residual norm and stop test; x += alpha u
// of the previous iteration; u = r + beta u with beta = res^2 / prev^2 (PRE:
// u = D^-1 r + beta u with beta = rz / prev rz); c = R A P u and the partials
// of dot(u, c).  The stop decision is recomputed from the partials each time,
// so it needs no flag: after a stop the partials are frozen and it[1 - par]
// repeats the count; alpha is then zero, so x is not changed again.
//
// A needs P u on the tile and a one-point halo.  The tile's own part is the
// block transform of its own u.  A halo point needs N = LEV + 2 coarse rows
// and columns of the neighbour's u, which the tile forms itself from r and
// the previous u (the neighbours' 4 x 16 x N values per component and one
// N x N corner block; the previous and the new u are double-buffered by
// parity, so no tile reads what another writes).  Every value adds its terms
// in the order of the block transform, so it has the neighbour's bits.  With
// the direction in a launch of its own, P u went through memory and the
// iteration had a third kernel boundary (at least 2.5 us on this chip).
// u and c are zero off the wavelet masks by construction (b, and with it r, u
// and D^-1, are).
template <bool PRE, int LEV, int FOLD, bool BIG>
__device__ __forceinline__ bool cg_step_tile(const CGArgs &a, int par, const int L)
{
    using T = double;
    __shared__ OpLds<T> s;
    __shared__ double lds[20];  // a slot per sum
    const GridDims &g = a.g;
    if (L >= g.nbx * g.nby) return false;
    int bx, by;
    band_tile(g, L, bx, by);
    const CGLayout &Lo = a.Lo;
    CgTile<LEV, BIG> t;
    t.place(Lo, bx * TILE, by * TILE);
    const unsigned at = t.at;
    const double2 *R = Lo.pair(CG_R), *P = Lo.pair(CG_P + par), *D = Lo.pair(CG_DINV);
    // loads in the order of first use: scalars and partials, the tile's
    // vectors, the coarse halo, the coefficients
    const int it = cg_scalar(&a.st->it[par]);
    const double told = cg_scalar(&a.st->tol), prev_res = cg_scalar(&a.st->res[1 - par]);
    const T alpha = cg_scalar(&a.st->alpha);
    double rz = 0.0, prev_rz = 0.0;
    LaneFold<FOLD> fr, fz;
    fr.load(a.Pr, g.npart);
    if constexpr (PRE) {
        prev_rz = cg_scalar(&a.st->rz[1 - par]);
        fz.load(a.Pz, g.npart);
    }
    const double2 r = elem<BIG>(R, at), p = elem<BIG>(P, at), x = elem<BIG>(Lo.pair(CG_X), at);
    const double2 dz = PRE ? elem<BIG>(D, at) : make_double2(0.0, 0.0);
    t.mb = elem<BIG>(Lo.M, at);
    t.place_halo(Lo);
    const double2 nr0 = elem<BIG>(R, t.h0), np0 = elem<BIG>(P, t.h0), nd0 = PRE ? elem<BIG>(D, t.h0) : make_double2(0.0, 0.0);
    const double2 nr1 = elem<BIG>(R, t.h1), np1 = elem<BIG>(P, t.h1), nd1 = PRE ? elem<BIG>(D, t.h1) : make_double2(0.0, 0.0);
    t.load_coef(Lo);
    double res;
    if constexpr (PRE) {
        double r2 = fr.sum(a.Pr, g.npart);
        rz = fz.sum(a.Pz, g.npart);
        tree256x2_open(r2, rz, lds);
        res = sqrt(r2);
    } else {
        res = sqrt(tree256_open(fr.sum(a.Pr, g.npart), lds));
    }
    double tol;
    if (it == 0) {
        const double abstol = a.tol_coarse * sqrt(tree256_open(lane_fold(a.Pb, g.npart), lds + 8));
        tol = a.reltol * res;
        if (abstol > tol) tol = abstol;
    } else {
        tol = told;
    }
    const bool done = (it >= a.maxiter) || (res <= tol);
    if (threadIdx.x == 0) {
        if (it == 0) a.st->tol = tol;
        a.st->res[par] = res;
        if constexpr (PRE) a.st->rz[par] = rz;
        if (done) {
            a.st->done = 1;
            a.st->iters = it;
            a.st->it[1 - par] = it;
            if (L == 0) {
                a.hflag->iters = it;
                a.hflag->done = 1;
            }
        }
    }
    if (alpha != 0.0) elem<BIG>(Lo.pair(CG_X), at) = make_double2(x.x + alpha * p.x, x.y + alpha * p.y);
    if (done) return true;
    const T beta = cg_beta<PRE>(it, res, prev_res, rz, prev_rz);
    const double2 un = cg_direction<PRE>(beta, r, p, dz);
    elem<BIG>(Lo.pair(CG_P + 1 - par), at) = un;
    double2 c;
    (void)t.apply(a.rdx, a.rdy, un, cg_direction<PRE>(beta, nr0, np0, nd0), cg_direction<PRE>(beta, nr1, np1, nd1), s, c,
                  [] { return true; });
    elem<BIG>(Lo.pair(CG_Q), at) = c;
    double du = un.x * c.x, dv = un.y * c.y;
    tree256x2_open(du, dv, lds + 12);
    if (threadIdx.x == 0) {
        if (bx < g.nbxu && by < g.nbyu) a.Pd[bx + g.nbxu * by] = du;
        if (bx < g.nbxv && by < g.nbyv) a.Pd[g.nbxu * g.nbyu + bx + g.nbxv * by] = dv;
    }
    return false;
}

// part 2: alpha = res^2 / dot(u, c) (PRE: rz / dot(u, c)), left for the next
// k_cg_step's x += alpha u; r -= alpha c, partials of ||r||^2 (PRE: and of
// (r, D^-1 r)) and the iteration count.  After a stop alpha is set to zero.
// EARLY: and nothing else is done.  Otherwise a launch after a stop stores r,
// its partials and the count unchanged (selected by the flag, which is then
// needed only at the stores), so that the flag's round trip does not precede
// the loads.
template <bool PRE, bool EARLY, int FOLD, bool BIG>
__device__ __forceinline__ void cg_update_tile(const CGArgs &a, int par, const int L)
{
    __shared__ double lds[20];  // a slot per sum
    const GridDims &g = a.g;
    if (L >= g.nbx * g.nby) return;
    if (EARLY && a.st->done) {
        if (threadIdx.x == 0) a.st->alpha = 0.0;
        return;
    }
    const bool stopped = !EARLY && cg_scalar(&a.st->done) != 0;
    int bx, by;
    band_tile(g, L, bx, by);
    const unsigned at = a.Lo.at(bx * TILE + (threadIdx.x & 15), by * TILE + (threadIdx.x >> 4));
    const int it = cg_scalar(&a.st->it[par]);
    const double res = cg_scalar(&a.st->res[par]);
    LaneFold<FOLD> fd;
    fd.load(a.Pd, g.npart);
    const double2 r = elem<BIG>(a.Lo.pair(CG_R), at), q = elem<BIG>(a.Lo.pair(CG_Q), at);
    const double2 dz = PRE ? elem<BIG>(a.Lo.pair(CG_DINV), at) : make_double2(0.0, 0.0);
    double rzc = 0.0;
    if constexpr (PRE) rzc = cg_scalar(&a.st->rz[par]);
    const double dot = tree256_open(fd.sum(a.Pd, g.npart), lds);
    const double alpha = (PRE ? rzc : res * res) / dot;
    if (threadIdx.x == 0) {
        a.st->it[1 - par] = stopped ? it : it + 1;
        a.st->alpha = stopped ? 0.0 : alpha;
    }
    double2 rn = make_double2(r.x - alpha * q.x, r.y - alpha * q.y);
    if (stopped) rn = r;
    elem<BIG>(a.Lo.pair(CG_R), at) = rn;
    double r2u = rn.x * rn.x, r2v = rn.y * rn.y, z2u = 0.0, z2v = 0.0;
    tree256x2_open(r2u, r2v, lds + 4);
    if constexpr (PRE) {
        z2u = rn.x * (dz.x * rn.x);
        z2v = rn.y * (dz.y * rn.y);
        tree256x2_open(z2u, z2v, lds + 12);
    }
    if (threadIdx.x == 0) {
        if (bx < g.nbxu && by < g.nbyu) {
            a.Pr[bx + g.nbxu * by] = r2u;
            if constexpr (PRE) a.Pz[bx + g.nbxu * by] = z2u;
        }
        if (bx < g.nbxv && by < g.nbyv) {
            const int q2 = g.nbxu * g.nbyu + bx + g.nbxv * by;
            a.Pr[q2] = r2v;
            if constexpr (PRE) a.Pz[q2] = z2v;
        }
    }
}

template <bool PRE, int LEV, int FOLD, bool BIG>
__global__ void __launch_bounds__(256) k_cg_step(CGArgs a, int par)
{
    (void)cg_step_tile<PRE, LEV, FOLD, BIG>(a, par, xcd_tile(a.nblk));
}

template <bool PRE, bool EARLY, int FOLD, bool BIG>
__global__ void __launch_bounds__(256) k_cg_update(CGArgs a, int par)
{
    cg_update_tile<PRE, EARLY, FOLD, BIG>(a, par, xcd_tile(a.nblk));
}

// Diagonal of the coarse-CG operator A_c = M_w R M_i A M_i P M_w
// (update_preconditioners.jl:73, with the masks the CG applies) at the
// points k of the wavelet masks: e_k' A_c e_k = phi' M_i A M_i phi with
// phi = P e_k, the Haar basis function of k, which is separable
// (Py (x) Px, from the inverse-transform rows of c_haar) and lives in k's
// Haar block, inside k's tile.  Workgroup (tile, component, coarse row ky)
// stages phi for each coarse column kx with a zero halo, evaluates the
// operator at the tile's points and sums phi (A phi) (FP64, canonical
// tree).  Writes 1 / |diagonal| (0 where the diagonal is 0 or off the
// masks) and, if diag is given, the diagonal.  Grid: (tiles, 32).
__global__ void __launch_bounds__(256) k_coarse_diag(GridDims g, OpCoef<double> c, const uint8_t *mwu,
                                                     const uint8_t *mwv, int levels, double *dinvu, double *dinvv,
                                                     double *diagu, double *diagv)
{
    __shared__ OpTile<double> s;
    __shared__ double lds[8];
    const int L = blockIdx.x;
    const int comp = blockIdx.y & 1, ky = blockIdx.y >> 1;
    const int bx = L % g.nbx, by = L / g.nbx;
    const bool has = comp == 0 ? (bx < g.nbxu && by < g.nbyu) : (bx < g.nbxv && by < g.nbyv);
    const int nxw = comp == 0 ? g.nxu : g.nxv, nyw = comp == 0 ? g.nyu : g.nyv;
    const int i0 = bx * TILE, j0 = by * TILE;
    if (!has || j0 + ky >= nyw) return;  // the whole workgroup
    const int lx = threadIdx.x & 15, ly = threadIdx.x >> 4;
    const int B = 2 << levels;
    PointCoef<double> pc;
    point_prefetch_op(g, c, i0 + lx, j0 + ly, comp == 0, comp == 1, pc);
    CellCoef<double> c0, c1;
    cell_prefetch(g, c, i0, j0, threadIdx.x, c0);
    cell_prefetch(g, c, i0, j0, threadIdx.x + 256, c1);
    const bool live = comp == 0 ? (pc.oku && pc.ui) : (pc.okv && pc.vi);
    // y factor of phi at this thread's row
    const int jb = ly & ~(B - 1), kjb = ky & ~(B - 1);
    double fy = 0.0;
    if (jb == kjb && j0 + ly < nyw) {
        const int my = min(nyw - (j0 + jb), B), col = ky - kjb;
        const uint32_t nz = c_haar[levels].nz[my][ly - jb], ng = c_haar[levels].neg[my][ly - jb];
        if ((nz >> col) & 1u) fy = ((ng >> col) & 1u) ? -1.0 : 1.0;
    }
    const int ib = lx & ~(B - 1);
    const int mx = i0 + lx < nxw ? min(nxw - (i0 + ib), B) : 0;
    const uint32_t nzx = mx > 0 ? c_haar[levels].nz[mx][lx - ib] : 0u;
    const uint32_t ngx = mx > 0 ? c_haar[levels].neg[mx][lx - ib] : 0u;
    // zero windows (the halo and the other component stay zero)
    for (int q = threadIdx.x; q < 18 * 19; q += 256) {
        (&s.U[0][0])[q] = 0.0;
        (&s.V[0][0])[q] = 0.0;
    }
    const uint8_t *mw = comp == 0 ? mwu : mwv;
    for (int kx = 0; kx < TILE && i0 + kx < nxw; ++kx) {
        const int kib = kx & ~(B - 1), col = kx - kib;
        double fx = 0.0;
        if (ib == kib && ((nzx >> col) & 1u)) fx = ((ngx >> col) & 1u) ? -1.0 : 1.0;
        const double phi = live ? fx * fy : 0.0;
        __syncthreads();  // previous intermediates read
        if (comp == 0)
            s.U[ly + 1][lx + 1] = phi;
        else
            s.V[ly + 1][lx + 1] = phi;
        __syncthreads();
        cell_compute(c, c0, threadIdx.x, s);
        cell_compute(c, c1, threadIdx.x + 256, s);
        __syncthreads();
        double v = 0.0;
        if (phi != 0.0) v = phi * (comp == 0 ? optile_u(c, s, pc, lx, ly) : optile_v(c, s, pc, lx, ly));
        v = tree256(v, lds);
        if (threadIdx.x == 0) {
            const int k = (i0 + kx) + nxw * (j0 + ky);
            const double d = mw[k] ? v : 0.0;
            (comp == 0 ? dinvu : dinvv)[k] = d != 0.0 ? 1.0 / fabs(d) : 0.0;
            if (diagu) (comp == 0 ? diagu : diagv)[k] = d;
        }
    }
}

// The whole coarse CG of a small grid in one workgroup (after k_cg_setup):
// the workgroup runs each part of an iteration on every tile in turn, so
// the barrier between two tiles stands in for the kernel boundary.  Tiles
// read only what earlier parts wrote and write only their own points,
// partials and parity slots, so the results are those of the two
// launches per iteration, bit for bit.  Ends at the stop, which every
// thread of every tile decides alike from the same partials and scalars,
// after maxiter + 1 iterations at most.  only_if: run only if it is set
// (the resident CG below gave up; what it starts from is still in place).
template <bool PRE, int LEV, bool BIG>
__global__ void __launch_bounds__(256) k_cg_solve1(CGArgs a, const int *only_if)
{
    if (only_if) {
        if (*only_if == 0) return;
        if (threadIdx.x == 0) a.hflag->gave_up = 1;
    }
    const int ntile = a.g.nbx * a.g.nby;
    for (int q = 0; q <= a.maxiter; ++q) {
        const int par = q & 1;
        bool stop = false;
        for (int L = 0; L < ntile; ++L) {
            stop = cg_step_tile<PRE, LEV, 1, BIG>(a, par, L);
            __syncthreads();
        }
        if (stop) break;
        for (int L = 0; L < ntile; ++L) {
            cg_update_tile<PRE, true, 1, BIG>(a, par, L);
            __syncthreads();
        }
    }
}

// Copies of the folded sums, in lines of their own: with one copy all
// wavefronts poll one line (3,564 of them at 1280 x 160), and the polls queue up.
constexpr int X_COPIES = 64, X_COPY = 32;  // ... and words from one to the next

// What the workgroups of the resident CG exchange, in tagged words (xput).
struct CGExchange {
    xword *c;       // c at every point: four planes of ns words (u, v), arena index, so that a
                    // wavefront stores and a row of the halo loads whole lines
    xword *pd;      // partials of (u, c): two words per partial
    xword *pr;      // partials of ||r||^2, then (Jacobi) of (r, D^-1 r)
    xword *root;    // the folded sums, if one workgroup folds, X_COPIES times: (u, c) at 0, the residual's at 8
    int *abort;     // a wait ran out
    unsigned tag;   // tag of iteration 0, larger than any used before
    unsigned limit; // polls of one wait
};

// The whole FP64 coarse CG in one launch, a tile per workgroup, all of them
// resident on the chip at once (after k_cg_setup; the host sees to it that
// they fit).  Everything a tile owns (r, u, x, the coefficients, the coarse
// halo's r and u) stays in registers; an iteration exchanges the partials of
// (u, c) and ||r||^2, and c with the neighbours, which advance the halo's r
// with it, so that the halo travels with the first sum and the second is
// alone.  The same operations in the same order as the launches': the same
// bits.
//
// What bounds it: two exchanges through the memory side of the chip and the
// latency of one tile's chain of seven LDS passes.  FLAT: every workgroup folds
// the partials itself (one hop).  Otherwise a workgroup without a tile does and
// publishes the sums (two hops).  An exchange among 6 / 63 / 246 / 891
// workgroups was measured at 1.2 / 2.0 / 2.7 / 18 us folding everywhere and
// 1.75 / 2.3 / 3.5 us for the last three folding once.  Measured per iteration,
// launches -> resident: 9.7 -> 5.4 us at 12 tiles, 9.5 -> 7.1 us at 63, 11.0 ->
// 8.5 us at 246, 13.6 -> 10.8 us at 441.  Two
// workgroups fit on a CU (165 to 193 registers).  With 128 registers four would,
// for up to 1016 tiles, but 16 to 52 of them spill: 20 us at 891 tiles against
// 18.6 us of the launches.
//
// Waits end: a wait that runs out of polls, or sees another's abort, raises
// the abort flag and the whole workgroup returns at its next check.  A check
// reads a flag that is written only in the waits before the barrier that
// precedes it, so a workgroup's threads agree.  x leaves for CG_Q at the stop
// and the arena is not written before, so k_cg_solve1 can start over.
// The sums that the set-up left.
template <bool PRE, int FOLD>
__device__ __forceinline__ void cg_resident_sums(const CGArgs &a, double *lds, double &sum0, double &sum1, double &abstol)
{
    LaneFold<FOLD> f0, f1;
    f0.load(a.Pr, a.g.npart);
    if constexpr (PRE) f1.load(a.Pz, a.g.npart);
    sum0 = f0.sum(a.Pr, a.g.npart);
    sum1 = 0.0;
    if constexpr (PRE) {
        sum1 = f1.sum(a.Pz, a.g.npart);
        tree256x2_open(sum0, sum1, lds);
    } else {
        sum0 = tree256_open(sum0, lds);
    }
    abstol = a.tol_coarse * sqrt(tree256(lane_fold(a.Pb, a.g.npart), lds + 8));
}

// The workgroup that folds: waits for all partials of a sum and publishes it.
template <bool PRE, int FOLD>
__device__ __forceinline__ void cg_resident_fold(const CGArgs &a, const CGExchange &E, double *lds, int *bad)
{
    const int np = a.g.npart;
    double sum0, sum1, abstol, tol = 0.0;
    cg_resident_sums<PRE, FOLD>(a, lds, sum0, sum1, abstol);
    for (int it = 0;; ++it) {
        const unsigned tag = E.tag + (unsigned)it;
        const double res = sqrt(sum0);
        if (it == 0) {
            tol = a.reltol * res;
            if (abstol > tol) tol = abstol;
        }
        if (it >= a.maxiter || res <= tol) return;
        XFold<FOLD> f, fz;
        f.want(true, np);
        for (unsigned n = 0;; ++n) {
            f.load(E.pd);
            if (f.check(tag)) break;
            if (x_give_up(n, E.limit, E.abort)) {
                bad[0] = 1;
                break;
            }
        }
        const double dot = tree256_open(f.sum(np), lds + 12);
        if (bad[0]) return;
        if (threadIdx.x < X_COPIES) xput2(E.root + X_COPY * threadIdx.x, tag, dot);
        f.want(true, np);
        fz.want(PRE, np);
        for (unsigned n = 0;; ++n) {
            f.load(E.pr);
            if constexpr (PRE) fz.load(E.pr + 2 * np);
            if (f.check(tag) & fz.check(tag)) break;
            if (x_give_up(n, E.limit, E.abort)) {
                bad[1] = 1;
                break;
            }
        }
        sum0 = f.sum(np);
        if constexpr (PRE) {
            sum1 = fz.sum(np);
            tree256x2_open(sum0, sum1, lds);
        } else {
            sum0 = tree256_open(sum0, lds);
        }
        if (bad[1]) return;
        if (threadIdx.x < X_COPIES) {
            xput2(E.root + X_COPY * threadIdx.x + 8, tag, sum0);
            if constexpr (PRE) xput2(E.root + X_COPY * threadIdx.x + 10, tag, sum1);
        }
    }
}

template <bool PRE, int LEV, bool FLAT>
__global__ void __launch_bounds__(256, 2) k_cg_resident(CGArgs a, CGExchange E)
{
    using T = double;
    constexpr int K = PRE ? 2 : 1, FOLD = FLAT ? 1 : 4;
    __shared__ OpLds<T> s;
    __shared__ double lds[36];  // a slot per sum
    __shared__ int bad[2];      // a wait of the first, second exchange ran out
    const GridDims &g = a.g;
    if (threadIdx.x < 2) bad[threadIdx.x] = 0;
    if (!FLAT && (int)blockIdx.x >= a.nblk) {
        if ((int)blockIdx.x == a.nblk) cg_resident_fold<PRE, FOLD>(a, E, lds, bad);
        return;
    }
    const int L = xcd_tile(a.nblk);
    if (L >= g.nbx * g.nby) return;
    int bx, by;
    band_tile(g, L, bx, by);
    const int np = g.npart;
    const CGLayout &Lo = a.Lo;
    CgTile<LEV> t;
    t.place(Lo, bx * TILE, by * TILE);
    t.place_halo(Lo);
    double sum0, sum1, abstol;
    cg_resident_sums<PRE, FOLD>(a, lds, sum0, sum1, abstol);
    // the tile's state; zero where there is no neighbour
    const double2 *R = Lo.pair(CG_R), *D = Lo.pair(CG_DINV);
    const double2 zero = make_double2(0.0, 0.0);
    double2 r = elem32(R, t.at), x = elem32(Lo.pair(CG_X), t.at), u = zero;
    double2 nr0 = elem32(R, t.h0), nr1 = elem32(R, t.h1), nu0 = zero, nu1 = zero;
    const double2 dz = PRE ? elem32(D, t.at) : zero, nd0 = PRE ? elem32(D, t.h0) : zero, nd1 = PRE ? elem32(D, t.h1) : zero;
    t.mb = elem32(Lo.M, t.at);
    t.load_coef(Lo);
    const bool west = bx > 0, east = bx + 1 < g.nbx, south = by > 0, north = by + 1 < g.nby;
    const bool have0 = t.rows ? (t.after ? north : south) : (t.after ? east : west);
    const bool have1 = t.corner ? (t.after ? east && south : west && north) : (t.l < 16 && have0);
    const bool has_u = bx < g.nbxu && by < g.nbyu, has_v = bx < g.nbxv && by < g.nbyv;
    const int pu = bx + g.nbxu * by, pv = g.nbxu * g.nbyu + bx + g.nbxv * by;
    const xword *root = E.root + X_COPY * ((4 * L + t.w) & (X_COPIES - 1));
    double tol = 0.0, prev_res = 1.0, prev_rz = 1.0, alpha = 0.0;
    for (int it = 0;; ++it) {
        const unsigned tag = E.tag + (unsigned)it;
        const double res = sqrt(sum0), rz = sum1;
        if (it == 0) {
            tol = a.reltol * res;
            if (abstol > tol) tol = abstol;
        }
        if (alpha != 0.0) x = make_double2(x.x + alpha * u.x, x.y + alpha * u.y);
        if (it >= a.maxiter || res <= tol) {
            elem32(Lo.pair(CG_Q), t.at) = x;
            if (L == 0 && threadIdx.x == 0) {
                a.hflag->iters = it;
                a.hflag->done = 1;
            }
            return;
        }
        const double beta = cg_beta<PRE>(it, res, prev_res, rz, prev_rz);
        u = cg_direction<PRE>(beta, r, u, dz);
        nu0 = cg_direction<PRE>(beta, nr0, nu0, nd0);
        nu1 = cg_direction<PRE>(beta, nr1, nu1, nd1);
        double2 c;
        if (!t.apply(a.rdx, a.rdy, u, nu0, nu1, s, c, [&] { return bad[1] == 0; })) return;
        {
            xword *q = &elem32(E.c, t.at);
            xput2(q, tag, c.x, Lo.ns);
            xput2(q + 2 * (size_t)Lo.ns, tag, c.y, Lo.ns);
        }
        double du = u.x * c.x, dv = u.y * c.y;
        tree256x2_open(du, dv, lds + 12);
        if (threadIdx.x == 0) {
            if (has_u) xput2(E.pd + 2 * pu, tag, du);
            if (has_v) xput2(E.pd + 2 * pv, tag, dv);
        }
        // first exchange: the halo's c and the sum
        double2 nc0 = zero, nc1 = zero;
        double dot;
        {
            XWait<4> w0, w1;
            XFold<FOLD> wf;
            XWait<2> wr;
            w0.want(have0);
            w1.want(have1);
            wf.want(FLAT, np);
            wr.want(!FLAT);
            for (unsigned n = 0;; ++n) {
                if (FLAT || n > 0) {  // two hops take longer than one: the halo is looked for after the first poll
                    w0.load(&elem32(E.c, t.h0), Lo.ns);
                    w1.load(&elem32(E.c, t.h1), Lo.ns);
                }
                if constexpr (FLAT) wf.load(E.pd);
                if constexpr (!FLAT) wr.load(root);
                const bool ok = w0.check(tag) & w1.check(tag) & wf.check(tag) & wr.check(tag);
                if (ok) break;
                if (x_give_up(n, E.limit, E.abort)) {
                    bad[0] = 1;
                    break;
                }
            }
            if (have0) nc0 = make_double2(w0.value(0), w0.value(1));
            if (have1) nc1 = make_double2(w1.value(0), w1.value(1));
            if constexpr (FLAT)
                dot = tree256_open(wf.sum(np), lds + 20);
            else
                dot = wr.value(0);
        }
        alpha = (PRE ? rz : res * res) / dot;
        prev_res = res;
        prev_rz = rz;
        r = make_double2(r.x - alpha * c.x, r.y - alpha * c.y);
        nr0 = make_double2(nr0.x - alpha * nc0.x, nr0.y - alpha * nc0.y);
        nr1 = make_double2(nr1.x - alpha * nc1.x, nr1.y - alpha * nc1.y);
        double r2u = r.x * r.x, r2v = r.y * r.y, z2u = 0.0, z2v = 0.0;
        tree256x2_open(r2u, r2v, lds + 4);
        if constexpr (PRE) {
            z2u = r.x * (dz.x * r.x);
            z2v = r.y * (dz.y * r.y);
            tree256x2_open(z2u, z2v, lds + 28);
        }
        if (bad[0]) return;
        if (threadIdx.x == 0) {
            if (has_u) {
                xput2(E.pr + 2 * pu, tag, r2u);
                if constexpr (PRE) xput2(E.pr + 2 * (np + pu), tag, z2u);
            }
            if (has_v) {
                xput2(E.pr + 2 * pv, tag, r2v);
                if constexpr (PRE) xput2(E.pr + 2 * (np + pv), tag, z2v);
            }
        }
        // second exchange: the residual norm
        {
            XFold<FOLD> wf, wz;
            XWait<2 * K> wr;
            wf.want(FLAT, np);
            wz.want(PRE && FLAT, np);
            wr.want(!FLAT);
            bool lost = false;
            for (unsigned n = 0;; ++n) {
                if constexpr (FLAT) wf.load(E.pr);
                if constexpr (FLAT && PRE) wz.load(E.pr + 2 * np);
                if constexpr (!FLAT) wr.load(root + 8);
                const bool ok = wf.check(tag) & wz.check(tag) & wr.check(tag);
                if (ok) break;
                if (x_give_up(n, E.limit, E.abort)) {
                    bad[1] = 1;
                    lost = true;
                    break;
                }
            }
            if constexpr (FLAT) {
                sum0 = wf.sum(np);
                if constexpr (PRE) {
                    sum1 = wz.sum(np);
                    tree256x2_open(sum0, sum1, lds);
                } else {
                    sum0 = tree256_open(sum0, lds);
                }
            } else {
                sum0 = lost ? __builtin_nan("") : wr.value(0);  // NaN does not stop the loop before its check
                if constexpr (PRE) sum1 = wr.value(1);
            }
        }
    }
}

// ===========================================================================
// Mixed-precision coarse CG: the Chronopoulos-Gear form of CG (one combined
// reduction per iteration) on FP32 vectors, with FP32 sums inside a
// workgroup and FP64 sums across workgroups and FP64 scalars, one launch per
// iteration.  In exact arithmetic it produces the iterates of the CG above;
// launch k computes
//     p = r + beta p,  s = w + beta s,  x += alpha p,  r -= alpha s,
//     w = A_c r,  gamma = (r, r),  delta = (w, r),
//     beta = gamma / gamma_old,  alpha = gamma / (delta - beta gamma / alpha_old).
// w = R A P r needs P r on the tile and on a one-point halo around it.  The
// tile's own part is the block transform of its own r (the Haar blocks never
// cross a tile).  The halo belongs to the neighbours' rings (their outermost
// rows and columns), where every workgroup stores the exact images P r, P w
// and P s of its own vectors at the end of each launch; the next launch forms
// the halo of P r_new = P r - alpha (P w + beta P s) from them, one linear
// step from exact values.  The rings, the partials and the scalars are
// double-buffered: the launch of parity PAR reads set PAR and writes set
// 1 - PAR, so no workgroup reads what another workgroup of the same launch
// writes.
//
// Layout: as the FP64 CG's arena in FP32: (u, v) pairs in zero-padded 2-D
// arrays shared by the u grid, the v grid and the h cells, point (i, j) at
// (i + 16) + px (j + 1), px = 16 (nbx + 1), so that a tile's rows are whole
// aligned 128-byte lines and windows, halos and tile stores need no bounds
// tests (what a tile stores past the end of a grid is zero).

struct CGMState {
    double igamma;  // 1 / ||r||^2 at the start of the launch that wrote this state
    double alpha;   // that launch's step length
    double ialpha;  // 1 / alpha
    double tol2;    // square of the stopping tolerance, fixed at iteration 0
    int it;         // iterations done
    int done;       // stop decided
};

struct CGMScalars {
    CGMState s[2];  // by launch parity
    int done;       // sticky stop flag, read by the host only
    int iters;      // iterations at the stop
    int abort;      // a workgroup of k_cgm_resident gave up waiting
};

// Arena arrays: (u, v) pairs, ns points each; then the corners' h*eta_av.
enum CGMPair {
    CGM_R = 0,       // residual r
    CGM_W = 1,       // w = A_c r
    CGM_P = 2,       // search direction p
    CGM_S = 3,       // s = A_c p
    CGM_X = 4,       // solution
    CGM_H = 5,       // thickness on u and v points, 0 off the masks
    CGM_B = 6,       // beta_eff on u and v points, 0 off the masks
    CGM_CELL = 7,    // per h cell: (h*eta_av, dimp)
    CGM_DINV = 8,    // Jacobi-preconditioned CG: 1 / |diag(A_c)|, 0 off the wavelet masks
    CGM_NPAIR = 9
};

// Ring images, compact per tile: for each parity and tile (ntile + 1 tiles,
// the last one all zero and never written, standing in for tiles past the
// edge) 64 slots: the tile's bottom row (y = 0, slots 0-15 by x), top row
// (y = 15, 16-31), left column (x = 0, 32-47 by y) and right column (x = 15,
// 48-63).  A slot holds (P r, P s) of u and v as one float4 and P w as one
// float2, so a side of a neighbour's halo is 16 consecutive ones of each.
struct CGMRings {
    float4 *rs;  // (P r)_u, (P r)_v, (P s)_u, (P s)_v
    float2 *w;   // (P w)_u, (P w)_v
};

__device__ __forceinline__ unsigned ring_at(int par, int ntile, int tile)
{
    return (unsigned)(par * (ntile + 1) + tile) * 64u;
}

// The ring slots of tile position (x, y): a row slot and a column slot, -1
// where there is none (a corner has two).
struct RingSlots {
    int row, col;
    __device__ __forceinline__ RingSlots(int x, int y)
    {
        row = y == 0 ? x : (y == 15 ? 16 + x : -1);
        col = x == 0 ? 32 + y : (x == 15 ? 48 + y : -1);
    }
    template <typename V>
    __device__ __forceinline__ void put(V *R, V v) const
    {
        if (row >= 0) R[row] = v;
        if (col >= 0) R[col] = v;
    }
    __device__ __forceinline__ void put_shared(xword *R, xword v) const
    {
        if (row >= 0) __hip_atomic_store(R + row, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (col >= 0) __hip_atomic_store(R + col, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
};

struct CGMLayout {
    float2 *F;      // pair array A at F + A * ns, then the corners (ns floats)
    uint8_t *M;     // mask bits (CB_*)
    unsigned px;    // row pitch
    unsigned ns;    // array stride
    __device__ __forceinline__ unsigned at(int i, int j) const
    {
        return (unsigned)(i + TILE) + __umul24(px, (unsigned)(j + 1));
    }
    // (dx, dy) from index k, dy >= -1 (as CGLayout::from)
    __device__ __forceinline__ unsigned from(unsigned k, int dx, int dy) const
    {
        return (k - px) + (unsigned)dx + __umul24(px, (unsigned)(dy + 1));
    }
    __device__ __forceinline__ float2 *pair(int a) const { return F + (size_t)a * ns; }
    __device__ __forceinline__ float *corner() const { return reinterpret_cast<float *>(F + (size_t)CGM_NPAIR * ns); }
};

// What the set-up and the end of the mixed CG read and write: the compact
// arrays.
struct CGMArgs {
    GridDims g;
    OpCoef<float> c;
    CGMLayout Lo;
    int levels;
    const uint8_t *mwu, *mwv;
    const float *bu, *bv;    // right-hand side
    float *xu, *xv;          // warm start in, solution out
    const float *t0u, *t0v;  // P x0
    const double *dinvu, *dinvv;  // Jacobi: 1 / |diag(A_c)|
    float *eu, *ev;          // the V-cycle's correction, += P x
    CGMRings R;
    double *Pb;              // partials of ||b||^2 per u / v block
    CGMScalars *st;
    CGMHostFlag *hflag;      // host-mapped stop report, reset here
    int nblk;
    int resident;            // the CG ran as k_cgm_resident
};

// setup (P x0 computed beforehand): r0 = b - R A P x0, p = s = 0, x = x0, the
// coefficients and mask bits into the arena, P r0 into the rings of set 0,
// partials of ||b||^2; resets the scalars.
template <bool PRE>
__global__ void __launch_bounds__(256) k_cgm_setup(CGMArgs a)
{
    __shared__ OpLds<float> s;
    __shared__ double lds[8];
    const GridDims &g = a.g;
    const int L = xcd_tile(a.nblk);
    if (L >= g.nbx * g.nby) return;
    if (L == 0 && threadIdx.x == 0) {
        for (int p = 0; p < 2; ++p) {
            a.st->s[p].igamma = 0.0;
            a.st->s[p].alpha = 0.0;
            a.st->s[p].ialpha = 0.0;
            a.st->s[p].tol2 = 0.0;
            a.st->s[p].it = 0;
            a.st->s[p].done = 0;
        }
        a.st->done = 0;
        a.st->iters = 0;
        a.st->abort = 0;
        a.hflag->done = 0;
        a.hflag->iters = 0;
        a.hflag->gave_up = 0;
    }
    int bx, by;
    const int tile_id = band_tile(g, L, bx, by);
    const bool has_u = bx < g.nbxu && by < g.nbyu, has_v = bx < g.nbxv && by < g.nbyv;
    const int i0 = bx * TILE, j0 = by * TILE;
    const int lx = threadIdx.x & 15, ly = threadIdx.x >> 4;
    OpOwn<float> o;
    op_own_index(g, i0 + lx, j0 + ly, o.oku, o.okv, o.ku, o.kv);
    const float bu = ld_or(o.oku, a.bu, o.ku, 0.f), bv = ld_or(o.okv, a.bv, o.kv, 0.f);
    const float xu = ld_or(o.oku, (const float *)a.xu, o.ku, 0.f), xv = ld_or(o.okv, (const float *)a.xv, o.kv, 0.f);
    // Jacobi: the rings hold P D^-1 r and ||b||^2 is the D^-1 norm
    const float dzu = PRE ? (float)fmin(ld_or(o.oku, a.dinvu, o.ku, 0.0), 1e30) : 1.f;  // finite in FP32
    const float dzv = PRE ? (float)fmin(ld_or(o.okv, a.dinvv, o.kv, 0.0), 1e30) : 1.f;
    const OpCoef<float> &c = a.c;
    op_restrict_tile(g, c, MaskSep<true>{c.ui, c.um, c.vi, c.vm, a.mwu, a.mwv}, a.levels, a.t0u, a.t0v, i0, j0, s, o);
    TilePair<float> &t = s.h.t, &m = s.h.m;
    const float ru = o.oku ? bu - ((o.mu & MB_WAVELET) ? t[0][ly][lx] : 0.f) : 0.f;
    const float rv = o.okv ? bv - ((o.mv & MB_WAVELET) ? t[1][ly][lx] : 0.f) : 0.f;
    const unsigned at = a.Lo.at(i0 + lx, j0 + ly);
    elem32(a.Lo.pair(CGM_R), at) = make_float2(ru, rv);
    elem32(a.Lo.pair(CGM_P), at) = make_float2(0.f, 0.f);
    elem32(a.Lo.pair(CGM_S), at) = make_float2(0.f, 0.f);
    elem32(a.Lo.pair(CGM_X), at) = make_float2(xu, xv);
    elem32(a.Lo.pair(CGM_H), at) = make_float2(o.hu, o.hv);
    elem32(a.Lo.pair(CGM_B), at) = make_float2(o.bu, o.bv);
    elem32(a.Lo.pair(CGM_CELL), at) = make_float2(o.heta, o.dimp);
    if constexpr (PRE) elem32(a.Lo.pair(CGM_DINV), at) = make_float2(dzu, dzv);
    elem32(a.Lo.corner(), at) = o.hetac;
    elem32(a.Lo.M, at) = (uint8_t)(((o.mu & MB_INNER) ? CB_INNER_U : 0) | ((o.mv & MB_INNER) ? CB_INNER_V : 0) |
                           ((o.mu & MB_WAVELET) ? CB_WAVELET_U : 0) | ((o.mv & MB_WAVELET) ? CB_WAVELET_V : 0));
    double b2u = PRE ? (double)bu * ((double)dzu * (double)bu) : (double)bu * (double)bu;
    double b2v = PRE ? (double)bv * ((double)dzv * (double)bv) : (double)bv * (double)bv;
    // each thread rewrites only its own entry; the transform ended with a barrier
    t[0][ly][lx] = (o.mu & MB_WAVELET) ? (PRE ? dzu * ru : ru) : 0.f;
    t[1][ly][lx] = (o.mv & MB_WAVELET) ? (PRE ? dzv * rv : rv) : 0.f;
    __syncthreads();
    haar_pair<false, float>(a.levels, t, m);
    RingSlots(lx, ly).put(a.R.rs + ring_at(0, g.nbx * g.nby, tile_id),
                          make_float4((o.mu & MB_INNER) ? t[0][ly][lx] : 0.f, (o.mv & MB_INNER) ? t[1][ly][lx] : 0.f, 0.f, 0.f));
    tree256x2(b2u, b2v, lds);
    if (threadIdx.x == 0) {
        if (has_u) a.Pb[bx + g.nbxu * by] = b2u;
        if (has_v) a.Pb[g.nbxu * g.nbyu + bx + g.nbxv * by] = b2v;
    }
}

// The end of the mixed CG: x back into the compact warm start, and e += P x
// at the inner points.
__global__ void __launch_bounds__(256) k_cgm_finish(CGMArgs a)
{
    const int L = xcd_tile(a.nblk);
    if (L >= a.g.nbx * a.g.nby) return;
    int bx, by;
    band_tile(a.g, L, bx, by);
    const unsigned at = a.Lo.at(bx * TILE + (int)(threadIdx.x & 15), by * TILE + (int)(threadIdx.x >> 4));
    const bool resident = a.resident && a.st->abort == 0;  // the resident CG leaves x in CGM_W
    const float2 x = elem32(a.Lo.pair(resident ? CGM_W : CGM_X), at);
    cg_finish_tile<float>(a.g, a.levels, bx, by, x.x, x.y, elem32(a.Lo.M, at), a.xu, a.xv, a.eu, a.ev);
}

// Block Haar transforms of 16-point lines held one point per lane (pos = the
// point's position in the line, blocks of B = 2^(LEV+1) points) as the
// butterflies that compose wavelet_matrix (src/Wavelets/update_wavelets.jl:
// 38-89).  A pair is (o, e = o + h) with o a multiple of 2h.
//   P (inverse), h = B/2 .. 1:           y_o = x_o - x_e,  y_e = x_o + x_e
//   R (transposed inverse), h = 1 .. B/2: y_o = x_o + x_e,  y_e = x_e - x_o
// Points past the end of the grid must hold zero: a pair whose e lies past
// the end then leaves x_o unchanged, as wavelet_matrix does for a partial
// block, and the garbage left in those points never reaches a point in range.
// Two lines at once (the u and the v tile), each stage one v_fmac_f32 with a
// DPP source per line, v += sign * partner(v) with sign in {-1, 0, +1}: the
// product is exact, so the fused multiply-add rounds exactly as the addition
// would.  Every block starts with two wait states: a DPP read of a register
// that the previous VALU instruction wrote needs them, and the compiler
// does not see the VALU writes inside these blocks.  The H = 4 partner is
// row_half_mirror of quad_perm [0,0,0,0], two DPP steps.
#define WAVI_DPP_TAIL " row_mask:0xf bank_mask:0xf bound_ctrl:1"

template <int H>
__device__ __forceinline__ void haar_stage_dpp(float &v0, float &v1, float sg)
{
    if constexpr (H == 1)
        asm("s_nop 1\n\tv_fmac_f32_dpp %0, %0, %2 quad_perm:[1,0,3,2]" WAVI_DPP_TAIL
            "\n\tv_fmac_f32_dpp %1, %1, %2 quad_perm:[1,0,3,2]" WAVI_DPP_TAIL
            : "+v"(v0), "+v"(v1) : "v"(sg));
    else if constexpr (H == 2)
        asm("s_nop 1\n\tv_fmac_f32_dpp %0, %0, %2 quad_perm:[2,3,0,1]" WAVI_DPP_TAIL
            "\n\tv_fmac_f32_dpp %1, %1, %2 quad_perm:[2,3,0,1]" WAVI_DPP_TAIL
            : "+v"(v0), "+v"(v1) : "v"(sg));
    else if constexpr (H == 8)
        asm("s_nop 1\n\tv_fmac_f32_dpp %0, %0, %2 row_ror:8" WAVI_DPP_TAIL
            "\n\tv_fmac_f32_dpp %1, %1, %2 row_ror:8" WAVI_DPP_TAIL
            : "+v"(v0), "+v"(v1) : "v"(sg));
    else {
        float t0, t1;
        asm("s_nop 1\n\tv_mov_b32_dpp %2, %0 quad_perm:[0,0,0,0]" WAVI_DPP_TAIL
            "\n\tv_mov_b32_dpp %3, %1 quad_perm:[0,0,0,0]" WAVI_DPP_TAIL
            "\n\ts_nop 1\n\tv_fmac_f32_dpp %0, %2, %4 row_half_mirror" WAVI_DPP_TAIL
            "\n\tv_fmac_f32_dpp %1, %3, %4 row_half_mirror" WAVI_DPP_TAIL
            : "+v"(v0), "+v"(v1), "=&v"(t0), "=&v"(t1) : "v"(sg));
    }
}

template <int H>
__device__ __forceinline__ float haar_sign_P(int pos)
{
    return ((pos & (H - 1)) == 0) ? ((pos & H) ? 1.f : -1.f) : 0.f;
}

template <int H>
__device__ __forceinline__ float haar_sign_R(int pos)
{
    return ((pos & (H - 1)) == 0) ? ((pos & H) ? -1.f : 1.f) : 0.f;
}

template <int LEV>
__device__ __forceinline__ void haar_lines_P(float &v0, float &v1, int pos)
{
    if constexpr (LEV >= 3) haar_stage_dpp<8>(v0, v1, haar_sign_P<8>(pos));
    if constexpr (LEV >= 2) haar_stage_dpp<4>(v0, v1, haar_sign_P<4>(pos));
    if constexpr (LEV >= 1) haar_stage_dpp<2>(v0, v1, haar_sign_P<2>(pos));
    haar_stage_dpp<1>(v0, v1, haar_sign_P<1>(pos));
}

template <int LEV>
__device__ __forceinline__ void haar_lines_R(float &v0, float &v1, int pos)
{
    haar_stage_dpp<1>(v0, v1, haar_sign_R<1>(pos));
    if constexpr (LEV >= 1) haar_stage_dpp<2>(v0, v1, haar_sign_R<2>(pos));
    if constexpr (LEV >= 2) haar_stage_dpp<4>(v0, v1, haar_sign_R<4>(pos));
    if constexpr (LEV >= 3) haar_stage_dpp<8>(v0, v1, haar_sign_R<8>(pos));
}

// Sum over a 16-lane row in FP32, left in every lane of the row.
__device__ __forceinline__ float row_sum16f(float v)
{
    v = v + dpp_f<DPP_XOR1>(v);
    v = v + dpp_f<DPP_XOR2>(v);
    v = v + dpp_f<DPP_HALF_MIRROR>(v);
    v = v + dpp_f<DPP_MIRROR>(v);
    return v;
}

struct CGMIterArgs {
    CGMLayout Lo;
    CGMRings R;
    float2 *Pgd;            // [2][npad]: per tile (r, r) and (w, r) partials by parity (0 past the tiles)
    CGMScalars *st;
    CGMHostFlag *hflag;     // host-mapped stop report
    const double *Pb;       // partials of ||b||^2 per u / v block
    GridDims g;
    int npad;               // partials per parity, a multiple of 1024
    float rdx, rdy;
    double tol_coarse, reltol;
    int maxiter, nblk;
};

template <bool PRE>
struct CgmSmem {
    float2 UV[18][19];               // window of P r (u and v points)
    float2 H[18][19];                // thickness window, 0 off the masks
    float4 cell[17][18];             // r_xx, r_yy, r_xy and the implicit term
    float2 T[2][TILE][TILE + 1];     // transposes of the block transforms
    float2 dz[PRE ? TILE : 1][TILE + 1];  // Jacobi: 1 / |diag(A_c)| of the tile
    uint8_t mb[TILE][TILE + 4];      // mask bits of the tile
    double red0[8];
    float red1[8];
    double red2[8];
};

// A thread's part of a tile in the mixed CG: its position, coefficients and
// what the tile does with a new r and s.
template <int LEV, bool PRE>
struct CgmTile {
    int tid, l, w, lx, ly, cx, cy;   // (lx, ly) row-major, (cx, cy) column-major (transposes)
    unsigned at0, at, mb;
    bool halo;
    int hx, hy;                      // its halo point of the window
    int ntl, hslot;                  // ... in the neighbour's ring (tile ntile: none)
    int ex, ey;                      // its cell before the tile (wavefront 0)
    float2 dz, hH, oH, cc, ec, oB;
    float ch, eh;

    __device__ __forceinline__ void place(const CGMLayout &Lo, int bx, int by)
    {
        tid = threadIdx.x;
        l = tid & 63;
        w = __builtin_amdgcn_readfirstlane(tid >> 6);
        lx = tid & 15;
        ly = tid >> 4;
        cx = tid >> 4;
        cy = tid & 15;
        // (24-bit products: a 32-bit multiply-add is emitted as a 64-bit one whose
        // unused high addend can be a register with a load in flight)
        at0 = Lo.at(bx * TILE, by * TILE);
        at = at0 + (unsigned)lx + __umul24(Lo.px, (unsigned)ly);
        const bool corner = w == 2 && l < 2;  // lane 0: (17, 0), of which u is read; lane 1: (0, 17), v
        halo = w == 3 || corner;
        hx = l == 0 ? 17 : 0;
        hy = l == 0 ? 0 : 17;
        ntl = hslot = 0;
        dz = make_float2(1.f, 1.f);
        hH = ec = make_float2(0.f, 0.f);
        eh = 0.f;
    }
    // Wavefronts 2 and 3: halo point (hx, hy) of the window from the
    // neighbours' rings: slot hslot of the tile ntl, (bx + hdx, by + hdy)
    __device__ __forceinline__ void place_halo(const GridDims &g, int bx, int by)
    {
        const int q = l & 15, side = l >> 4;
        int hdx = l == 0 ? 1 : -1, hdy = -hdx;
        hslot = l == 0 ? 16 : 15;
        if (w == 3) {
            halo_side(l, hx, hy);
            hdx = side == 0 ? -1 : (side == 1 ? 1 : 0);
            hdy = side == 2 ? -1 : (side == 3 ? 1 : 0);
            hslot = q + (side == 0 ? 48 : (side == 1 ? 32 : (side == 2 ? 16 : 0)));
        }
        const int nbxx = bx + hdx, nbyy = by + hdy;
        ntl = (nbxx >= 0 && nbxx < g.nbx && nbyy >= 0 && nbyy < g.nby) ? nbxx + g.nbx * nbyy : g.nbx * g.nby;
    }
    __device__ __forceinline__ float2 load(const CGMLayout &Lo, int A, unsigned k) const
    {
        return elem32((const float2 *)Lo.pair(A), k);
    }
    __device__ __forceinline__ float2 halo_thickness(const CGMLayout &Lo) const
    {
        return load(Lo, CGM_H, Lo.from(at0, hx - 1, hy - 1));
    }
    __device__ __forceinline__ void load_coef(const CGMLayout &Lo)
    {
        oH = load(Lo, CGM_H, at);
        cc = load(Lo, CGM_CELL, at);
        ch = elem32((const float *)Lo.corner(), at);
        // the cells before the tile: (0, 0..16), (1..16, 0); lanes past them repeat the last
        ex = l < 17 ? 0 : (l < 33 ? l - 16 : 16);
        ey = l < 17 ? l : 0;
        float2 c = make_float2(0.f, 0.f);
        float h = 0.f;
        if (w == 0) {
            const unsigned ea = Lo.from(at0, ex - 1, ey - 1);
            c = load(Lo, CGM_CELL, ea);
            h = elem32((const float *)Lo.corner(), ea);
        }
        ec = c;
        eh = h;
        oB = load(Lo, CGM_B, at);
    }
    // From r and s1 (S: there is one) of the tile and the halo's P r (hv): the
    // own point's w = R A P r and P w, and P r, P s of the point (cx, cy),
    // given to `images` as soon as they are known.
    template <bool S, class Images>
    __device__ __forceinline__ void operate(float rdx, float rdy, float2 r, float2 s1, float2 hv, CgmSmem<PRE> &sm,
                                            float2 &wn, float2 &pw, Images images)
    {
        const bool inu = mb & CB_INNER_U, inv = mb & CB_INNER_V, mwu = mb & CB_WAVELET_U, mwv = mb & CB_WAVELET_V;
        // ---- x pass of P r and P s (Jacobi: of D^-1 r and D^-1 s); halo and
        // thickness windows into LDS
        {
            float a0 = mwu ? (PRE ? dz.x * r.x : r.x) : 0.f, a1 = mwv ? (PRE ? dz.y * r.y : r.y) : 0.f;
            haar_lines_P<LEV>(a0, a1, lx);
            sm.T[0][ly][lx] = make_float2(a0, a1);
            if (S) {
                float a2 = mwu ? (PRE ? dz.x * s1.x : s1.x) : 0.f, a3 = mwv ? (PRE ? dz.y * s1.y : s1.y) : 0.f;
                haar_lines_P<LEV>(a2, a3, lx);
                sm.T[1][ly][lx] = make_float2(a2, a3);
            }
        }
        sm.mb[ly][lx] = (uint8_t)mb;
        if constexpr (PRE) sm.dz[ly][lx] = dz;
        sm.H[ly + 1][lx + 1] = oH;
        if (halo) {
            sm.UV[hy][hx] = hv;
            sm.H[hy][hx] = hH;
        }
        __syncthreads();
        // ---- y pass in the column-major lanes: P r into the window, rings of P r
        // and P s
        {
            const unsigned m = sm.mb[cy][cx];
            const float2 t0 = sm.T[0][cy][cx];
            float y0 = t0.x, y1 = t0.y;
            haar_lines_P<LEV>(y0, y1, cy);
            const float2 pr = make_float2((m & CB_INNER_U) ? y0 : 0.f, (m & CB_INNER_V) ? y1 : 0.f);
            sm.UV[cy + 1][cx + 1] = pr;
            float2 ps = make_float2(0.f, 0.f);
            if (S) {
                const float2 t1 = sm.T[1][cy][cx];
                float y2 = t1.x, y3 = t1.y;
                haar_lines_P<LEV>(y2, y3, cy);
                ps = make_float2((m & CB_INNER_U) ? y2 : 0.f, (m & CB_INNER_V) ? y3 : 0.f);
            }
            images(pr, ps);
        }
        __syncthreads();
        // ---- intermediates of the cell (x, y) of the 17 x 17 window, whose own
        // point has the value uv and the thickness h
        auto intermediates = [&](int x, int y, float2 uv, float2 h, float2 hd, float hc) -> float4 {
            const float u1 = sm.UV[y][x + 1].x, v1 = sm.UV[y + 1][x].y;
            const float2 d = sm.UV[y + 1][x + 1];
            const float dudx = rdx * (u1 - uv.x), dvdy = rdy * (v1 - uv.y);
            const float divq = rdx * (sm.H[y][x + 1].x * u1 - h.x * uv.x) + rdy * (sm.H[y + 1][x].y * v1 - h.y * uv.y);
            return make_float4(2.f * hd.x * (2.f * dudx + dvdy), 2.f * hd.x * (2.f * dvdy + dudx),
                               hc * (rdy * (d.x - u1) + rdx * (d.y - v1)), hd.y * divq);
        };
        const float2 uv = sm.UV[ly + 1][lx + 1];
        const float4 own = intermediates(lx + 1, ly + 1, uv, oH, cc, ch);
        if (w == 0) sm.cell[ey][ex] = intermediates(ex, ey, sm.UV[ey][ex], sm.H[ey][ex], ec, eh);
        sm.cell[ly + 1][lx + 1] = own;
        __syncthreads();
        // ---- A at the tile's points (zero off the inner masks), R x pass
        {
            const float4 left = sm.cell[ly + 1][lx], below = sm.cell[ly][lx + 1];
            const float rxy00 = sm.cell[ly][lx].z;
            const float d_rxx = rdx * (own.x - left.x);
            const float d_rxy_u = rdy * (left.z - rxy00);
            const float d_ext_u = rdx * (own.w - left.w);
            const float Au = ((d_rxx + d_rxy_u) - oB.x * uv.x) - oH.x * d_ext_u;
            const float d_ryy = rdy * (own.y - below.y);
            const float d_rxy_v = rdx * (below.z - rxy00);
            const float d_ext_v = rdy * (own.w - below.w);
            const float Av = ((d_ryy + d_rxy_v) - oB.y * uv.y) - oH.y * d_ext_v;
            float a0 = inu ? Au : 0.f, a1 = inv ? Av : 0.f;
            haar_lines_R<LEV>(a0, a1, lx);
            sm.T[0][ly][lx] = make_float2(a0, a1);
        }
        __syncthreads();
        // ---- R y pass, wavelet mask (w), P y pass
        {
            const float2 t0 = sm.T[0][cy][cx];
            float c0 = t0.x, c1 = t0.y;
            haar_lines_R<LEV>(c0, c1, cy);
            const unsigned m = sm.mb[cy][cx];
            const float2 wc = make_float2((m & CB_WAVELET_U) ? c0 : 0.f, (m & CB_WAVELET_V) ? c1 : 0.f);
            float q0 = wc.x, q1 = wc.y;
            if constexpr (PRE) {
                const float2 d = sm.dz[cy][cx];
                q0 = d.x * wc.x;
                q1 = d.y * wc.y;
            }
            haar_lines_P<LEV>(q0, q1, cy);
            sm.T[0][cy][cx] = wc;
            sm.T[1][cy][cx] = make_float2(q0, q1);
        }
        __syncthreads();
        // ---- P x pass
        wn = sm.T[0][ly][lx];
        const float2 tq = sm.T[1][ly][lx];
        float tw_u = tq.x, tw_v = tq.y;
        haar_lines_P<LEV>(tw_u, tw_v, lx);
        pw = make_float2(inu ? tw_u : 0.f, inv ? tw_v : 0.f);
    }
    // The tile's partials (r, u) and (w, u) with u = D^-1 r under Jacobi, (r, r)
    // and (w, r) without; valid in thread 0 after its barrier.
    __device__ __forceinline__ float2 partials(float2 r, float2 wn, CgmSmem<PRE> &sm) const
    {
        const float zr_u = PRE ? dz.x * r.x : r.x, zr_v = PRE ? dz.y * r.y : r.y;
        float gg = r.x * zr_u + r.y * zr_v;
        float dd = wn.x * zr_u + wn.y * zr_v;
        gg = wave_total_rows_f(row_sum16f(gg));
        dd = wave_total_rows_f(row_sum16f(dd));
        if (l == 63) {
            sm.red1[w] = gg;
            sm.red1[4 + w] = dd;
        }
        __syncthreads();
        return make_float2((sm.red1[0] + sm.red1[1]) + (sm.red1[2] + sm.red1[3]),
                           (sm.red1[4] + sm.red1[5]) + (sm.red1[6] + sm.red1[7]));
    }
};

// alpha and beta of an iteration from the sums (r, r) and (w, r) of the one
// before (S: its state)
__device__ __forceinline__ void cgm_scalars(const CGMState &S, double gamma, double delta, double &alpha, double &beta)
{
    beta = S.it == 0 ? 0.0 : gamma * S.igamma;
    alpha = gamma / (S.it == 0 ? delta : delta - beta * gamma * S.ialpha);
}

// the state they leave
__device__ __forceinline__ CGMState cgm_next(const CGMState &S, double gamma, double alpha, double tol2)
{
    CGMState n;
    n.igamma = 1.0 / gamma;
    n.alpha = alpha;
    n.ialpha = 1.0 / alpha;
    n.tol2 = tol2;
    n.it = S.it + 1;
    n.done = 0;
    return n;
}

// square of the stopping tolerance, at iteration 0
template <bool PRE>
__device__ __forceinline__ double cgm_tol2(const CGMIterArgs &a, double gamma, CgmSmem<PRE> &sm)
{
    const double abstol = a.tol_coarse * sqrt(lanes_sum(a.Pb, a.g.npart, sm.red2));
    double tol = a.reltol * sqrt(gamma);
    if (abstol > tol) tol = abstol;
    return tol * tol;
}

// One iteration (INIT: the launch before the first iteration, which only
// computes w0 = A_c r0 and the rings of set 1: P r0, P s = 0, P w0, and the
// partial (r0, r0), (w0, r0)).  All loads are issued up front, unconditional
// in the padded layout, so that the memory round trip is paid once.  Seven
// barriers: partial sums; block transforms of r and s (x pass, transpose,
// y pass straight into the window); intermediates; operator and R x pass;
// R y pass and P y pass; P x pass and the new partials.
// PRE (inside the flexible CG's linear solves only): the Jacobi-
// preconditioned form with u = D^-1 r, w = A_c u, gamma = (r, u),
// delta = (w, u); D^-1 is pointwise, so u, D^-1 s and D^-1 w are formed
// where they are used and the rings hold P D^-1 r, P D^-1 s, P D^-1 w (the
// halo of P u_new is then the same linear step).
//
// Each operand is loaded and staged once: a thread loads the pairs of its
// own point and its own cell, wavefront 3 the halo's four sides, wavefront 2
// the two halo corners that are read, wavefront 0 the 33 cells before the
// tile; an h cell's four intermediates go through LDS as one float4.
template <int PAR, bool INIT, int LEV, bool PRE>
__device__ __forceinline__ bool cgm_iter_tile(const CGMIterArgs &a, const int L)
{
    static_assert(!INIT || PAR == 0, "the initial launch reads set 0");
    __shared__ CgmSmem<PRE> sm;
    const GridDims &g = a.g;
    const int ntile = g.nbx * g.nby;
    if (L >= ntile) return false;
    int bx, by;
    const int tile_id = band_tile(g, L, bx, by);
    constexpr int NP = 1 - PAR;
    // Launch q >= 1 performs iteration k = q - 1, so PAR == 0 iff k is odd.
    // x is advanced every other iteration: an even iteration leaves it, the
    // odd one after it applies both steps, x_{k+1} = x_{k-1} +
    // (alpha_{k-1} + alpha_k beta_k) p_{k-1} + alpha_k r_k, and a stop after
    // an even iteration applies the pending alpha_{k-1} p_{k-1}.
    constexpr bool XUPD = PAR == 0;
    const CGMLayout &Lo = a.Lo;
    CgmTile<LEV, PRE> t;
    t.place(Lo, bx, by);
    const int tid = t.tid;
    auto cstore = [&](int A, float2 v) {
        st_nt(reinterpret_cast<double *>(&elem32(Lo.pair(A), t.at)),
              __hiloint2double(__float_as_int(v.y), __float_as_int(v.x)));
    };
    // ---- loads, all issued before the first use, in the order they are
    // needed: the wait for a load also waits for every load issued before
    // it, so the partials come first and the coefficients last
    const CGMState S = a.st->s[PAR];
    // partials of the previous launch
    float2 pv[4];
    if (!INIT) {
#pragma unroll
        for (int e = 0; e < 4; ++e) pv[e] = a.Pgd[PAR * a.npad + tid + 256 * e];
    }
    t.mb = elem32((const uint8_t *)Lo.M, t.at);
    float2 r = t.load(Lo, CGM_R, t.at), w0 = make_float2(0.f, 0.f), p0 = w0, s0 = w0, x0 = w0;
    if (!INIT) {
        w0 = t.load(Lo, CGM_W, t.at);
        p0 = t.load(Lo, CGM_P, t.at);
        s0 = t.load(Lo, CGM_S, t.at);
        if (XUPD) x0 = t.load(Lo, CGM_X, t.at);
    }
    if constexpr (PRE) t.dz = t.load(Lo, CGM_DINV, t.at);
    const float2 dz = t.dz;
    float4 hrs = make_float4(0.f, 0.f, 0.f, 0.f);
    float2 hw = make_float2(0.f, 0.f), hH = hw;
    if (t.w >= 2) {
        t.place_halo(g, bx, by);
        const unsigned hr_at = ring_at(PAR, ntile, t.ntl) + (unsigned)t.hslot;
        hrs = elem32((const float4 *)a.R.rs, hr_at);
        if (!INIT) hw = elem32((const float2 *)a.R.w, hr_at);
        hH = t.halo_thickness(Lo);
    }
    t.hH = hH;
    t.load_coef(Lo);
    // ---- scalars from the previous launch's partials (FP64 across workgroups)
    float fa = 0.f, fb = 0.f, fxp = 0.f;
    if (!INIT) {
        double gamma = 0.0, delta = 0.0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            gamma = gamma + (double)pv[e].x;
            delta = delta + (double)pv[e].y;
        }
        for (int q = tid + 1024; q < a.npad; q += 256) {
            const float2 v = a.Pgd[PAR * a.npad + q];
            gamma = gamma + (double)v.x;
            delta = delta + (double)v.y;
        }
        wg_sum2(gamma, delta, sm.red0);
        if (S.done) {
            if (L == 0 && tid == 0) a.st->s[NP] = S;
            return true;
        }
        // stop when ||r|| <= tol, tested as ||r||^2 <= tol^2
        const double tol2 = S.it == 0 ? cgm_tol2<PRE>(a, gamma, sm) : S.tol2;
        if (S.it >= a.maxiter || gamma <= tol2) {
            if (L == 0 && tid == 0) {
                CGMState n = S;
                n.tol2 = tol2;
                n.done = 1;
                a.st->s[NP] = n;
                a.st->done = 1;
                a.st->iters = S.it;
                a.hflag->iters = S.it;
                a.hflag->done = 1;
            }
            if (XUPD && S.it > 0) {
                const float fp = (float)S.alpha;
                cstore(CGM_X, make_float2(x0.x + fp * p0.x, x0.y + fp * p0.y));
            }
            return true;
        }
        double alpha, beta;
        cgm_scalars(S, gamma, delta, alpha, beta);
        if (L == 0 && tid == 0) a.st->s[NP] = cgm_next(S, gamma, alpha, tol2);
        fa = (float)alpha;
        fb = (float)beta;
        fxp = XUPD ? (float)(S.alpha + alpha * beta) : 0.f;
    }
    // ---- vector updates on the tile (zero past the ends of the grids); with
    // Jacobi the direction and x take u = D^-1 r where they take r
    float2 s1 = make_float2(0.f, 0.f);
    if (!INIT) {
        const float z_u = PRE ? dz.x * r.x : r.x, z_v = PRE ? dz.y * r.y : r.y;
        const float p_u = z_u + fb * p0.x, p_v = z_v + fb * p0.y;
        if (XUPD) cstore(CGM_X, make_float2((x0.x + fxp * p0.x) + fa * z_u, (x0.y + fxp * p0.y) + fa * z_v));
        s1 = make_float2(w0.x + fb * s0.x, w0.y + fb * s0.y);
        r = make_float2(r.x - fa * s1.x, r.y - fa * s1.y);
        cstore(CGM_P, make_float2(p_u, p_v));
        cstore(CGM_S, s1);
        cstore(CGM_R, r);
    }
    const float2 hv = INIT ? make_float2(hrs.x, hrs.y)
                           : make_float2(hrs.x - fa * (hw.x + fb * hrs.z), hrs.y - fa * (hw.y + fb * hrs.w));
    float2 wn, pw;
    t.template operate<!INIT>(
        a.rdx, a.rdy, r, s1, hv, sm, wn, pw,
        [&](float2 pr, float2 ps) {
            RingSlots(t.cx, t.cy).put(a.R.rs + ring_at(NP, ntile, tile_id), make_float4(pr.x, pr.y, ps.x, ps.y));
        });
    cstore(CGM_W, wn);
    RingSlots(t.lx, t.ly).put(a.R.w + ring_at(NP, ntile, tile_id), pw);
    const float2 part = t.partials(r, wn, sm);
    if (tid == 0) a.Pgd[NP * a.npad + tile_id] = part;
    return false;
}

// One coarse-CG iteration of one CG problem (the tile of workgroup
// blockIdx.x, XCD-aware).
template <int PAR, bool INIT, int LEV, bool PRE>
__global__ void __launch_bounds__(256) k_cgm_iter(CGMIterArgs a)
{
    (void)cgm_iter_tile<PAR, INIT, LEV, PRE>(a, xcd_tile(a.nblk));
}

// The whole mixed coarse CG of a small grid in one workgroup (after
// k_cgm_setup): the initial launch's work and then each iteration on every
// tile in turn, the barrier between two tiles standing in for the kernel
// boundary.  A tile reads the other tiles' rings and partials of the
// previous iteration only, so the results are those of one launch per
// iteration, bit for bit.  Every thread decides the stop alike (same
// partials, same scalars); at most maxiter + 1 iterations.
template <int LEV, bool PRE>
__device__ __forceinline__ void cgm_solve1_run(const CGMIterArgs &a, const int *only_if)
{
    if (only_if) {  // the resident CG gave up; what it started from is still in place
        if (*only_if == 0) return;
        if (threadIdx.x == 0) a.hflag->gave_up = 1;
    }
    const int ntile = a.g.nbx * a.g.nby;
    for (int L = 0; L < ntile; ++L) {
        (void)cgm_iter_tile<0, true, LEV, PRE>(a, L);
        __syncthreads();
    }
    for (int q = 1; q <= a.maxiter + 1; ++q) {
        bool stop = false;
        for (int L = 0; L < ntile; ++L) {
            stop = (q & 1) ? cgm_iter_tile<1, false, LEV, PRE>(a, L) : cgm_iter_tile<0, false, LEV, PRE>(a, L);
            __syncthreads();
        }
        if (stop) break;
    }
}

template <int LEV, bool PRE>
__global__ void __launch_bounds__(256) k_cgm_solve1(CGMIterArgs a, const int *only_if)
{
    cgm_solve1_run<LEV, PRE>(a, only_if);
}

// What the workgroups of the resident mixed CG exchange, in tagged words.
struct CGMExchange {
    xword *ring;    // [2][6][tiles][64]: (P r)_u, (P r)_v, (P s)_u, (P s)_v, (P w)_u, (P w)_v of the ring slots
    xword *part;    // [2][tiles][2]: the partials (r, r) and (w, r)
    int *abort;     // a wait ran out
    unsigned tag;   // tag of the first exchange, larger than any used before
    unsigned limit; // polls of one wait
};

// The whole mixed coarse CG in one launch, a tile per workgroup, all of them
// resident at once (after k_cgm_setup; k_cg_resident tells of the waits).  r,
// w, p, s and x of a tile stay in registers; an iteration has one exchange: the
// tiles' two sums, which every workgroup folds, and the ring images of the
// neighbours, in two sets by parity, since a workgroup may be one exchange
// ahead of another.  The same operations in the same order as the launches':
// the same bits.
// At most 256 tiles, one partial per thread: measured per iteration, launches
// -> resident, 5.1 -> 3.5 us at 6 tiles, 5.2 -> 4.1 at 63, 5.9 -> 5.1 at 246.
// With two partials per thread 7.1 -> 9.2 us at 357; with one workgroup
// folding, as in FP64, 7.1 -> 7.2 us at 357 and 10.4 -> 10.1 at 891.
template <int LEV, bool PRE>
__device__ __forceinline__ void cgm_resident_tile(const CGMIterArgs &a, const CGMExchange &E, int blk)
{
    __shared__ CgmSmem<PRE> sm;
    __shared__ int bad;  // a wait ran out; checked after the barrier that follows the wait
    const GridDims &g = a.g;
    const int ntile = g.nbx * g.nby, tid = threadIdx.x;
    if (tid == 0) bad = 0;
    CGMState S{};
    const int L = (blk & 7) * (a.nblk >> 3) + (blk >> 3);
    if (L >= ntile) return;
    int bx, by;
    const int tile_id = band_tile(g, L, bx, by);
    const CGMLayout &Lo = a.Lo;
    CgmTile<LEV, PRE> t;
    t.place(Lo, bx, by);
    const float2 zero = make_float2(0.f, 0.f);
    t.mb = elem32((const uint8_t *)Lo.M, t.at);
    float2 r = t.load(Lo, CGM_R, t.at), x = t.load(Lo, CGM_X, t.at), w = zero, p = zero, s = zero;
    if constexpr (PRE) t.dz = t.load(Lo, CGM_DINV, t.at);
    float4 hrs = make_float4(0.f, 0.f, 0.f, 0.f);
    if (t.w >= 2) {
        t.place_halo(g, bx, by);
        hrs = elem32((const float4 *)a.R.rs, ring_at(0, ntile, t.ntl) + (unsigned)t.hslot);
        t.hH = t.halo_thickness(Lo);
    }
    t.load_coef(Lo);
    const bool want = t.halo && t.ntl < ntile;
    const size_t plane = (size_t)ntile * 64;
    const size_t from = (size_t)t.ntl * 64 + t.hslot;
    const RingSlots row_major(t.lx, t.ly), col_major(t.cx, t.cy);
    float2 hv = make_float2(hrs.x, hrs.y), pw;
    // images and sums of set par under a tag
    auto images = [&](int par, unsigned tag, float2 pr, float2 ps) {
        xword *R = E.ring + (size_t)(par * 6) * plane + (size_t)tile_id * 64;
        const xword h = (xword)tag << 32;
        col_major.put_shared(R, h | (unsigned)__float_as_int(pr.x));
        col_major.put_shared(R + plane, h | (unsigned)__float_as_int(pr.y));
        col_major.put_shared(R + 2 * plane, h | (unsigned)__float_as_int(ps.x));
        col_major.put_shared(R + 3 * plane, h | (unsigned)__float_as_int(ps.y));
    };
    auto sums = [&](int par, unsigned tag) {
        xword *R = E.ring + (size_t)(par * 6) * plane + (size_t)tile_id * 64;
        const xword h = (xword)tag << 32;
        row_major.put_shared(R + 4 * plane, h | (unsigned)__float_as_int(pw.x));
        row_major.put_shared(R + 5 * plane, h | (unsigned)__float_as_int(pw.y));
        const float2 part = t.partials(r, w, sm);
        if (tid == 0) {
            xword *P = E.part + (size_t)(par * ntile + tile_id) * 2;
            xput(P, tag, (unsigned)__float_as_int(part.x));
            xput(P + 1, tag, (unsigned)__float_as_int(part.y));
        }
    };
    t.template operate<false>(
        a.rdx, a.rdy, r, zero, hv, sm, w, pw, [&](float2 pr, float2 ps) { images(1, E.tag, pr, ps); });
    sums(1, E.tag);
    for (int q = 1;; ++q) {
        const unsigned tag = E.tag + (unsigned)(q - 1);
        const int par = q & 1;
        // the exchange
        double gamma, delta;
        XWait<6> wh;
        wh.want(want);
        {
            const xword *ring = E.ring + (size_t)(par * 6) * plane + from;
            XWait<2> wp;
            wp.want(tid < ntile);
            for (unsigned n = 0;; ++n) {
                wh.load(ring, plane);
                wp.load(E.part + (size_t)(par * ntile + tid) * 2);
                const bool ok = wh.check(tag) & wp.check(tag);
                if (ok) break;
                if (x_give_up(n, E.limit, E.abort)) {
                    bad = 1;
                    break;
                }
            }
            gamma = tid < ntile ? (double)__int_as_float((int)wp.v[0]) : 0.0;
            delta = tid < ntile ? (double)__int_as_float((int)wp.v[1]) : 0.0;
            wg_sum2(gamma, delta, sm.red0);
            if (bad) return;
        }
        const bool xupd = par == 0;
        const double tol2 = S.it == 0 ? cgm_tol2<PRE>(a, gamma, sm) : S.tol2;
        if (S.it >= a.maxiter || gamma <= tol2) {
            if (xupd && S.it > 0) {
                const float fp = (float)S.alpha;
                x = make_float2(x.x + fp * p.x, x.y + fp * p.y);
            }
            elem32(Lo.pair(CGM_W), t.at) = x;
            if (L == 0 && tid == 0) {
                a.hflag->iters = S.it;
                a.hflag->done = 1;
            }
            return;
        }
        double alpha, beta;
        cgm_scalars(S, gamma, delta, alpha, beta);
        const float fa = (float)alpha, fb = (float)beta;
        const float z_u = PRE ? t.dz.x * r.x : r.x, z_v = PRE ? t.dz.y * r.y : r.y;
        if (xupd) {
            const float fxp = (float)(S.alpha + alpha * beta);
            x = make_float2((x.x + fxp * p.x) + fa * z_u, (x.y + fxp * p.y) + fa * z_v);
        }
        S = cgm_next(S, gamma, alpha, tol2);
        p = make_float2(z_u + fb * p.x, z_v + fb * p.y);
        s = make_float2(w.x + fb * s.x, w.y + fb * s.y);
        r = make_float2(r.x - fa * s.x, r.y - fa * s.y);
        auto word = [&](int k) { return want ? __int_as_float((int)wh.v[k]) : 0.f; };
        hv = make_float2(word(0) - fa * (word(4) + fb * word(2)), word(1) - fa * (word(5) + fb * word(3)));
        t.template operate<true>(a.rdx, a.rdy, r, s, hv, sm, w, pw,
                                       [&](float2 pr, float2 ps) { images(1 - par, tag + 1, pr, ps); });
        sums(1 - par, tag + 1);
    }
}

template <int LEV, bool PRE>
__global__ void __launch_bounds__(256, 4) k_cgm_resident(CGMIterArgs a, CGMExchange E)
{
    cgm_resident_tile<LEV, PRE>(a, E, blockIdx.x);
}

// The same iteration of several independent CG problems (an ensemble's
// members, each with its own arena, rings, partials and scalars) in one
// launch.  Member m owns the workgroups first[m] .. first[m] + nblk_m - 1;
// every first[m] and nblk_m is a multiple of 8, so group_member, indexed by
// blockIdx.x / 8, names the member, and a member's workgroups map to its
// tiles exactly as k_cgm_iter's do (blockIdx.x mod 8 is preserved).
struct CGMBatch {
    const CGMIterArgs *members;
    const int *group_member;
    const int *first;
};

template <int PAR, bool INIT, int LEV, bool PRE>
__global__ void __launch_bounds__(256) k_cgm_iter_batch(CGMBatch B)
{
    const int m = B.group_member[blockIdx.x >> 3];
    const CGMIterArgs a = B.members[m];
    const int w = (int)blockIdx.x - B.first[m];
    (void)cgm_iter_tile<PAR, INIT, LEV, PRE>(a, (w & 7) * (a.nblk >> 3) + (w >> 3));
}

// The resident CGs of several problems in one launch; the workgroups of one
// exchange nothing with those of another, so each stops by itself.
template <int LEV, bool PRE>
__global__ void __launch_bounds__(256, 4) k_cgm_resident_batch(CGMBatch B, const CGMExchange *ex)
{
    const int m = B.group_member[blockIdx.x >> 3];
    const CGMIterArgs a = B.members[m];
    const CGMExchange E = ex[m];
    cgm_resident_tile<LEV, PRE>(a, E, (int)blockIdx.x - B.first[m]);
}

// ... and what stands in for those that gave up, a workgroup each.
template <int LEV, bool PRE>
__global__ void __launch_bounds__(256) k_cgm_solve1_batch(CGMBatch B, const CGMExchange *ex)
{
    const CGMIterArgs a = B.members[blockIdx.x];
    cgm_solve1_run<LEV, PRE>(a, ex[blockIdx.x].abort);
}

// out = mask_out ? H(mask_in ? in : 0) : 0 on the u grid (comp 0) and v grid
// mask[k] != 0 at a point ok of a tile, true there without a mask (mask ==
// nullptr), false where !ok.  The load is unconditional (a branch on the
// pointer would give it a wait of its own): without a mask it reads byte 0
// of `any`, a valid buffer, and ignores it.
__device__ __forceinline__ bool mask_or_all(const uint8_t *mask, const void *any, bool ok, int k)
{
    const bool has = mask != nullptr;
    const uint8_t *p = has ? mask : static_cast<const uint8_t *>(any);
    const uint8_t b = p[(ok & has) ? k : 0];
    return ok & (!has | (b != 0));  // no short circuit, which would branch around the load
}

// Haar transform (dir 0 forward, 1 inverse, 2 transposed inverse) of the
// masked u and v inputs into the masked outputs.
template <typename Tin, typename Tout>
__global__ void k_tile_haar(GridDims g, const HaarTable *tab, int levels, int dir,
                            const Tin *inu, const Tin *inv, const uint8_t *min_u, const uint8_t *min_v,
                            Tout *outu, Tout *outv, const uint8_t *mout_u, const uint8_t *mout_v)
{
    __shared__ TilePair<Tout> t, m;
    const int lx = threadIdx.x & 15, ly = threadIdx.x >> 4;
    const int bx = blockIdx.x, by = blockIdx.y;
    const int i0 = bx * TILE, j0 = by * TILE;
    const int i = i0 + lx, j = j0 + ly;
    const bool has_u = bx < g.nbxu && by < g.nbyu, has_v = bx < g.nbxv && by < g.nbyv;
    if (dir != 0) {
        // the +-1 transforms: the u and the v tile together, every input
        // and mask loaded first (ld_or)
        const int ku = i + g.nxu * j, kv = i + g.nxv * j;
        const bool oku = has_u && i < g.nxu && j < g.nyu, okv = has_v && i < g.nxv && j < g.nyv;
        const Tin xu = ld_or(oku, inu, ku, Tin(0)), xv = ld_or(okv, inv, kv, Tin(0));
        const bool iu = mask_or_all(min_u, inu, oku, ku), iv = mask_or_all(min_v, inv, okv, kv);
        const bool ou = mask_or_all(mout_u, inu, oku, ku), ov = mask_or_all(mout_v, inv, okv, kv);
        t[0][ly][lx] = (oku && iu) ? (Tout)xu : Tout(0);
        t[1][ly][lx] = (okv && iv) ? (Tout)xv : Tout(0);
        __syncthreads();
        if (dir == 1)
            haar_pair<false, Tout>(levels, t, m);
        else
            haar_pair<true, Tout>(levels, t, m);
        if (oku) outu[ku] = ou ? t[0][ly][lx] : Tout(0);
        if (okv) outv[kv] = ov ? t[1][ly][lx] : Tout(0);
        return;
    }
    if (has_u) {
        int k = i + g.nxu * j;
        bool ok = i < g.nxu && j < g.nyu;
        t[0][ly][lx] = (ok && (!min_u || min_u[k])) ? (Tout)inu[k] : Tout(0);
        __syncthreads();
        haar_tile<Tout>(tab, 0, t[0], m[0], i0, j0, g.nxu, g.nyu);
        if (ok) outu[k] = (!mout_u || mout_u[k]) ? t[0][ly][lx] : Tout(0);
        __syncthreads();
    }
    if (has_v) {
        int k = i + g.nxv * j;
        bool ok = i < g.nxv && j < g.nyv;
        t[0][ly][lx] = (ok && (!min_v || min_v[k])) ? (Tout)inv[k] : Tout(0);
        __syncthreads();
        haar_tile<Tout>(tab, 0, t[0], m[0], i0, j0, g.nxv, g.nyv);
        if (ok) outv[k] = (!mout_v || mout_v[k]) ? t[0][ly][lx] : Tout(0);
        __syncthreads();
    }
}

// update_velocities_on_h_grid! (update_state.jl:164-178) and update_dhdt!
// (:184-189)
__global__ void k_post_solve(GridDims g, const uint8_t *hm, const uint8_t *um, const uint8_t *vm,
                             const double *U, const double *V, const double *beta, const double *f1,
                             const double *f2, const double *hu, const double *hv, const double *acc,
                             const double *mel, double *uh, double *vh, double *ubo, double *vbo,
                             double *uso, double *vso, double *dhdt, double rdx, double rdy)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= g.nx * g.ny) return;
    const int i = k % g.nx, j = k / g.nx;
    const int nxu = g.nxu, nx = g.nx;
    // every load issued before the first store (which the compiler cannot
    // move them past) and before the mask is tested
    const int u1 = (i + 1) + nxu * j, u0 = i + nxu * j, v1 = i + nx * (j + 1), v0 = i + nx * j;
    const double U0 = U[u0], U1 = U[u1], V0 = V[v0], V1 = V[v1];
    const double bk = beta[k], f1k = f1[k], f2k = f2[k], acck = acc[k], melk = mel[k];
    const double hu0 = hu[u0], hu1 = hu[u1], hv0 = hv[v0], hv1 = hv[v1];
    const bool hk = hm[k], mu0 = um[u0], mu1 = um[u1], mv0 = vm[v0], mv1 = vm[v1];
    double u_ = 0.5 * U0 + 0.5 * U1;
    double v_ = 0.5 * V0 + 0.5 * V1;
    uh[k] = u_;
    vh[k] = v_;
    double ub = u_ / (1.0 + bk * f2k);
    double vb = v_ / (1.0 + bk * f2k);
    ubo[k] = ub;
    vbo[k] = vb;
    uso[k] = ub * (1.0 + bk * f1k);
    vso[k] = vb * (1.0 + bk * f1k);
    if (hk) {
        double q1 = mu1 ? hu1 * U1 : 0.0;
        double q0 = mu0 ? hu0 * U0 : 0.0;
        double p1 = mv1 ? hv1 * V1 : 0.0;
        double p0 = mv0 ? hv0 * V0 : 0.0;
        double div = (rdx * q1 - rdx * q0) + (rdy * p1 - rdy * p0);
        dhdt[k] = (acck - melk) - div;
    }
}

// update_thickness! (run_simulation.jl:24-42), evolveShelves = true
__global__ void k_update_thickness(int nh, const uint8_t *hm, const uint8_t *hfix, double *h, const double *dhdt,
                                   double hmin, double dt)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nh || !hm[k]) return;
    double a = hmin - h[k], b = dt * dhdt[k];
    double upd = a > b ? a : b;
    if (hfix[k]) upd = 0.0;
    h[k] = h[k] + upd;
}

// quad_f2 = h/(3 eta_av) on the h mask (src/Fields/HGrid.jl:229)
__global__ void k_init_quad_f2(int nh, const uint8_t *hm, const double *h, const double *etaav, double *f2)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < nh && hm[k]) f2[k] = h[k] / (3.0 * etaav[k]);
}

// device math probe: fn 0 det_pow(x, y), 1 sqrt(x), 2 x / y
__global__ void k_math_probe(int fn, const double *x, const double *y, double *out, int n)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    if (fn == 0) out[k] = det_pow(x[k], y[k]);
    else if (fn == 1) out[k] = sqrt(x[k]);
    else out[k] = x[k] / y[k];
}

}  // namespace wavi
