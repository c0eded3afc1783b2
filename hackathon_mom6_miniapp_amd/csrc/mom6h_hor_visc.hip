// mom6h_hor_visc.hip -- horizontal viscosity on gfx950.
//
// Arithmetic of src/serial/mom6_hor_visc_serial.F90:464-1109 with the
// Laplacian (constant Kh) and biharmonic (constant Ah) operators, free- or
// no-slip; and (k_hv_closures, further below) the Smagorinsky and Leith
// viscosities with the thickness-aware bounds.  One 3D launch computes every layer: each thread forms the
// strain/stress values its diffu/diffv stencil needs directly from u, v, h
// (no 2D work arrays, no per-layer launches).  On grids whose metric arrays
// are constant every operator runs as a march of waves along j instead
// (k_hv_march), bit-identical to the general kernels.
//
// The serial code keeps ONE 2D array for Kh (and Ah) at h- and q-points: the
// h-point pass writes is..ie x js..je but the stress uses is-1..ie+1 x
// js-1..je+1 (:744-819), so the ring takes what the previous layer's q-point
// pass left there (Kh_bg_xy on is-1..ie x js-1..je, zero elsewhere, and zero
// everywhere on the first layer of the first call).  Likewise Del2u/Del2v are
// only formed on their own ranges (:587-607) and read as zero outside.  Those
// values only reach diffu on column is-1 and ie and diffv on rows js-1 and je
// (biharmonic: also the first interior column/row), and are reproduced here.
#include "mom6h_fused.h"

#include <algorithm>
#include <initializer_list>
#include <utility>

namespace mom6h {

struct HV {
    Dims d;
    double Kh, Ah, h_neglect;
    int laplacian, biharmonic, no_slip, first_call;
    const double *DY_dxT, *DX_dyT, *DY_dxBu, *DX_dyBu, *IdyCu, *IdxCu, *IdyCv, *IdxCv;
    const double *IareaCu, *IareaCv, *mask2dT, *mask2dBu, *reduction_xx, *reduction_xy;
    const double *dy2h, *dx2h, *dy2q, *dx2q;
    const double *Idx2dyCu, *Idxdy2u, *Idx2dyCv, *Idxdy2v;
    const unsigned char *mask_bits;   // 0/1 masks, one byte per point (MomArgsT::mask)
    double *Del2u, *Del2v;
    // closures (the general kernel): Smagorinsky_Kh/_Ah, Leith_Kh/_Ah,
    // better_bound_Kh/_Ah = bound_Kh/_Ah (hor_visc_init :179-193)
    int smag_Kh, smag_Ah, leith_Kh, leith_Ah, bound;
    const double *areaT, *dxBu, *dyBu, *IdxBu, *IdyBu;
    double *ring_Kh, *ring_Ah;
};

// horizontal tension at an h point (:503-530)
__device__ inline double sh_xx_at(const HV &p, const double *u, const double *v, int i, int j, int k)
{
    const Dims &d = p.d;
    const double dudx = p.DY_dxT[IX2(d, i, j)] *
                        ((p.IdyCu[IX2(d, i, j)] * u[IX3(d, i, j, k)]) - (p.IdyCu[IX2(d, i - 1, j)] * u[IX3(d, i - 1, j, k)]));
    const double dvdy = p.DX_dyT[IX2(d, i, j)] *
                        ((p.IdxCv[IX2(d, i, j)] * v[IX3(d, i, j, k)]) - (p.IdxCv[IX2(d, i, j - 1)] * v[IX3(d, i, j - 1, k)]));
    return dudx - dvdy;
}

// shearing strain at a q point with the slip condition (:513-547)
__device__ inline double sh_xy_at(const HV &p, const double *u, const double *v, int I, int J, int k)
{
    const Dims &d = p.d;
    const double dvdx = p.DY_dxBu[IX2(d, I, J)] *
                        ((v[IX3(d, I + 1, J, k)] * p.IdyCv[IX2(d, I + 1, J)]) - (v[IX3(d, I, J, k)] * p.IdyCv[IX2(d, I, J)]));
    const double dudy = p.DX_dyBu[IX2(d, I, J)] *
                        ((u[IX3(d, I, J + 1, k)] * p.IdxCu[IX2(d, I, J + 1)]) - (u[IX3(d, I, J, k)] * p.IdxCu[IX2(d, I, J)]));
    const double m = p.mask2dBu[IX2(d, I, J)];
    return (p.no_slip ? (2.0 - m) : m) * (dvdx + dudy);
}

// Del2u / Del2v (:587-607) on their ranges, zero elsewhere (never written there).
__global__ void k_hv_del2(HV p, const double *__restrict__ u, const double *__restrict__ v)
{
    const Dims &d = p.d;
    const int i = d.isc - 1 + blockIdx.x * blockDim.x + threadIdx.x;
    const int j = d.jsc - 1 + blockIdx.y;
    const int k = 1 + blockIdx.z;
    if (i > d.iec) return;
    const long long c = IX3(d, i, j, k), c2 = IX2(d, i, j);
    if (j >= d.jsc) {
        p.Del2u[c] = p.Idx2dyCu[c2] * ((p.dx2q[c2] * sh_xy_at(p, u, v, i, j, k)) -
                                       (p.dx2q[IX2(d, i, j - 1)] * sh_xy_at(p, u, v, i, j - 1, k))) +
                     p.Idxdy2u[c2] * ((p.dy2h[IX2(d, i + 1, j)] * sh_xx_at(p, u, v, i + 1, j, k)) -
                                      (p.dy2h[c2] * sh_xx_at(p, u, v, i, j, k)));
    }
    if (i >= d.isc) {
        p.Del2v[c] = p.Idxdy2v[c2] * ((p.dy2q[c2] * sh_xy_at(p, u, v, i, j, k)) -
                                      (p.dy2q[IX2(d, i - 1, j)] * sh_xy_at(p, u, v, i - 1, j, k))) -
                     p.Idx2dyCv[c2] * ((p.dx2h[IX2(d, i, j + 1)] * sh_xx_at(p, u, v, i, j + 1, k)) -
                                       (p.dx2h[c2] * sh_xx_at(p, u, v, i, j, k)));
    }
}

// Kh or Ah seen at an h point of the stress ring (see the file comment).
__device__ inline double visc_h(const HV &p, double val, int i, int j, int k)
{
    const Dims &d = p.d;
    if (i >= d.isc && i <= d.iec && j >= d.jsc && j <= d.jec) return val;
    if (i >= d.isc - 1 && i <= d.iec && j >= d.jsc - 1 && j <= d.jec)
        return (k == 1 && p.first_call) ? 0.0 : val;
    return 0.0;
}

// str_xx * h (:807-895) at h point (i,j)
__device__ inline double str_xx_at(const HV &p, const double *u, const double *v, const double *h,
                                   int i, int j, int k)
{
    const Dims &d = p.d;
    const double sh = sh_xx_at(p, u, v, i, j, k);
    double str = p.laplacian ? -(visc_h(p, p.Kh, i, j, k) * sh) : 0.0;
    if (p.biharmonic) {
        const double d_del2u = (p.IdyCu[IX2(d, i, j)] * p.Del2u[IX3(d, i, j, k)]) -
                               (p.IdyCu[IX2(d, i - 1, j)] * p.Del2u[IX3(d, i - 1, j, k)]);
        const double d_del2v = (p.IdxCv[IX2(d, i, j)] * p.Del2v[IX3(d, i, j, k)]) -
                               (p.IdxCv[IX2(d, i, j - 1)] * p.Del2v[IX3(d, i, j - 1, k)]);
        const double d_str = visc_h(p, p.Ah, i, j, k) *
                             ((p.DY_dxT[IX2(d, i, j)] * d_del2u) - (p.DX_dyT[IX2(d, i, j)] * d_del2v));
        str = str + d_str;
    }
    return str * (h[IX3(d, i, j, k)] * p.reduction_xx[IX2(d, i, j)]);
}

// str_xy * hq (:954-1053) at q point (I,J)
__device__ inline double str_xy_at(const HV &p, const double *u, const double *v, const double *h,
                                   int I, int J, int k)
{
    const Dims &d = p.d;
    const long long c2 = IX2(d, I, J);
    const double sh = sh_xy_at(p, u, v, I, J, k);
    double str = p.laplacian ? -(p.Kh * sh) : 0.0;
    if (p.biharmonic) {
        const double d_str =
            p.Ah * ((p.DY_dxBu[c2] * ((p.Del2v[IX3(d, I + 1, J, k)] * p.IdyCv[IX2(d, I + 1, J)]) -
                                      (p.Del2v[IX3(d, I, J, k)] * p.IdyCv[c2]))) +
                    (p.DX_dyBu[c2] * ((p.Del2u[IX3(d, I, J + 1, k)] * p.IdxCu[IX2(d, I, J + 1)]) -
                                      (p.Del2u[IX3(d, I, J, k)] * p.IdxCu[c2]))));
        str = str + d_str;
    }
    const double hq = 0.25 * ((h[IX3(d, I, J, k)] + h[IX3(d, I + 1, J + 1, k)]) +
                              (h[IX3(d, I + 1, J, k)] + h[IX3(d, I, J + 1, k)]));
    if (p.no_slip) return str * (hq * p.reduction_xy[c2]);
    return str * (hq * p.mask2dBu[c2] * p.reduction_xy[c2]);
}

// diffu, diffv over the full data domain (zero outside their ranges, :486-494, :1059-1078)
__global__ void k_hv_main(HV p, const double *__restrict__ u, const double *__restrict__ v,
                          const double *__restrict__ h, double *__restrict__ diffu,
                          double *__restrict__ diffv)
{
    const Dims &d = p.d;
    const int i = d.isd + blockIdx.x * blockDim.x + threadIdx.x;
    const int j = d.jsd + blockIdx.y;
    const int k = 1 + blockIdx.z;
    if (i > d.ied) return;
    const long long c = IX3(d, i, j, k), c2 = IX2(d, i, j);
    double du = 0.0, dv = 0.0;
    if (i >= d.isc - 1 && i <= d.iec && j >= d.jsc && j <= d.jec) {
        const double h_u = 0.5 * (p.mask2dT[c2] * h[c] + p.mask2dT[IX2(d, i + 1, j)] * h[IX3(d, i + 1, j, k)]);
        du = ((p.IdxCu[c2] * ((p.dx2q[IX2(d, i, j - 1)] * str_xy_at(p, u, v, h, i, j - 1, k)) -
                              (p.dx2q[c2] * str_xy_at(p, u, v, h, i, j, k))) +
               p.IdyCu[c2] * ((p.dy2h[c2] * str_xx_at(p, u, v, h, i, j, k)) -
                              (p.dy2h[IX2(d, i + 1, j)] * str_xx_at(p, u, v, h, i + 1, j, k)))) *
              p.IareaCu[c2]) / (h_u + p.h_neglect);
    }
    if (i >= d.isc && i <= d.iec && j >= d.jsc - 1 && j <= d.jec) {
        const double h_v = 0.5 * (p.mask2dT[c2] * h[c] + p.mask2dT[IX2(d, i, j + 1)] * h[IX3(d, i, j + 1, k)]);
        dv = ((p.IdyCv[c2] * ((p.dy2q[IX2(d, i - 1, j)] * str_xy_at(p, u, v, h, i - 1, j, k)) -
                              (p.dy2q[c2] * str_xy_at(p, u, v, h, i, j, k))) -
               p.IdxCv[c2] * ((p.dx2h[c2] * str_xx_at(p, u, v, h, i, j, k)) -
                              (p.dx2h[IX2(d, i, j + 1)] * str_xx_at(p, u, v, h, i, j + 1, k)))) *
              p.IareaCv[c2]) / (h_v + p.h_neglect);
    }
    diffu[c] = du;
    diffv[c] = dv;
}

// ---------------------------------------------------------------------------
// The general kernel: Smagorinsky and Leith viscosities and the
// thickness-aware bounds (:612-1040).  The reference fills 2D work arrays per
// layer; here every value is a function of the layer's u, v, h evaluated where
// it is needed, with the reference's ranges: a work value outside the range
// its loop writes reads as the array's initial value (zero; hrat_min and
// visc_bound_rem: one).  The Kh and Ah arrays are shared between h and q
// points: the h-point pass writes is..ie x js..je, the q-point pass is-1..ie x
// js-1..je, and the stress at the h points of the ring (is-1..ie+1 x
// js-1..je+1 minus the interior) reads what the previous layer's q-point pass
// left there -- for the first layer, the previous call's last layer (ring_Kh,
// ring_Ah), zero elsewhere.

__device__ inline double sq(double x) { return x * x; }

// inv_PI3 = 1/(3.14159265358979_dp**3), inv_PI6 = 1/(3.14159265358979_dp**6)
// (:154-155), the integer powers by squaring as the compiled reference has them
#define HV_PI 3.14159265358979
#define HV_INV_PI3 (1.0 / ((HV_PI * HV_PI) * HV_PI))
#define HV_INV_PI6 (1.0 / (((HV_PI * HV_PI) * (HV_PI * HV_PI)) * (HV_PI * HV_PI)))

__device__ inline bool interior(const Dims &d, int i, int j)
{
    return i >= d.isc && i <= d.iec && j >= d.jsc && j <= d.jec;
}
__device__ inline bool q_range(const Dims &d, int I, int J)   // Isq..Ieq x Jsq..Jeq
{
    return I >= d.isc - 1 && I <= d.iec && J >= d.jsc - 1 && J <= d.jec;
}

__device__ inline double dvdx_at(const HV &p, const double *v, int I, int J, int k)
{
    const Dims &d = p.d;
    return p.DY_dxBu[IX2(d, I, J)] *
           ((v[IX3(d, I + 1, J, k)] * p.IdyCv[IX2(d, I + 1, J)]) - (v[IX3(d, I, J, k)] * p.IdyCv[IX2(d, I, J)]));
}
__device__ inline double dudy_at(const HV &p, const double *u, int I, int J, int k)
{
    const Dims &d = p.d;
    return p.DX_dyBu[IX2(d, I, J)] *
           ((u[IX3(d, I, J + 1, k)] * p.IdxCu[IX2(d, I, J + 1)]) - (u[IX3(d, I, J, k)] * p.IdxCu[IX2(d, I, J)]));
}

// Leith: vorticity at q points (:612-626) and its gradients (:629-645)
__device__ inline double vort_at(const HV &p, const double *u, const double *v, int I, int J, int k)
{
    const double m = p.mask2dBu[IX2(p.d, I, J)];
    return (p.no_slip ? (2.0 - m) : m) * (dvdx_at(p, v, I, J, k) - dudy_at(p, u, I, J, k));
}
__device__ inline double vort_dx_at(const HV &p, const double *u, const double *v, int i, int j, int k)
{
    const Dims &d = p.d;
    if (!interior(d, i, j)) return 0.0;
    const double DY_dxBu_loc = p.dyBu[IX2(d, i, j)] * p.IdxBu[IX2(d, i, j)];
    return DY_dxBu_loc * ((vort_at(p, u, v, i, j, k) * p.IdyCu[IX2(d, i, j)]) -
                          (vort_at(p, u, v, i - 1, j, k) * p.IdyCu[IX2(d, i - 1, j)]));
}
__device__ inline double vort_dy_at(const HV &p, const double *u, const double *v, int I, int j, int k)
{
    const Dims &d = p.d;
    if (!(I >= d.isc - 1 && I <= d.iec && j >= d.jsc && j <= d.jec)) return 0.0;
    const double DX_dyBu_loc = p.dxBu[IX2(d, I, j)] * p.IdyBu[IX2(d, I, j)];
    return DX_dyBu_loc * ((vort_at(p, u, v, I, j, k) * p.IdxCv[IX2(d, I, j)]) -
                          (vort_at(p, u, v, I, j - 1, k) * p.IdxCv[IX2(d, I, j - 1)]));
}
// Laplacian of the vorticity at q points (:648-659), zero outside Isq..Ieq x Jsq..Jeq
__device__ inline double del2vort_q_at(const HV &p, const double *u, const double *v, int I, int J, int k)
{
    const Dims &d = p.d;
    if (!q_range(d, I, J)) return 0.0;
    return p.DY_dxBu[IX2(d, I, J)] * ((vort_dx_at(p, u, v, I + 1, J, k) * p.IdyCv[IX2(d, I + 1, J)]) -
                                      (vort_dx_at(p, u, v, I, J, k) * p.IdyCv[IX2(d, I, J)])) +
           p.DX_dyBu[IX2(d, I, J)] * ((vort_dy_at(p, u, v, I, J + 1, k) * p.IdxCu[IX2(d, I, J + 1)]) -
                                      (vort_dy_at(p, u, v, I, J, k) * p.IdxCu[IX2(d, I, J)]));
}

// thickness at u and v points with the land mask (:551-562)
__device__ inline double h_u_at(const HV &p, const double *h, int I, int j, int k)
{
    const Dims &d = p.d;
    return 0.5 * (p.mask2dT[IX2(d, I, j)] * h[IX3(d, I, j, k)] + p.mask2dT[IX2(d, I + 1, j)] * h[IX3(d, I + 1, j, k)]);
}
__device__ inline double h_v_at(const HV &p, const double *h, int i, int J, int k)
{
    const Dims &d = p.d;
    return 0.5 * (p.mask2dT[IX2(d, i, J)] * h[IX3(d, i, J, k)] + p.mask2dT[IX2(d, i, J + 1)] * h[IX3(d, i, J + 1, k)]);
}
// hrat_min (:730-737) on is..ie x js..je, one elsewhere
__device__ inline double hrat_at(const HV &p, const double *h, int i, int j, int k)
{
    if (!interior(p.d, i, j)) return 1.0;
    const double h_min = fmin(fmin(fmin(h_u_at(p, h, i, j, k), h_u_at(p, h, i - 1, j, k)), h_v_at(p, h, i, j, k)),
                              h_v_at(p, h, i, j - 1, k));
    return fmin(1.0, h_min / (h[IX3(p.d, i, j, k)] + p.h_neglect));
}

// Kh and Ah at an interior h point (:743-863); *rem = visc_bound_rem
__device__ inline void visc_h_point(const HV &p, const double *u, const double *v, const double *h, int i, int j,
                                    int k, double *Kh_out, double *Ah_out)
{
    const Dims &d = p.d;
    const double a2 = p.areaT[IX2(d, i, j)];
    double shear = 0.0, vvm = 0.0, hrat = 1.0;
    if (p.smag_Kh || p.smag_Ah) {   // Shear_mag (:710-720)
        const double sh_xx_sq = sq(sh_xx_at(p, u, v, i, j, k));
        const double sh_xy_sq = 0.25 * ((sq(sh_xy_at(p, u, v, i - 1, j - 1, k)) + sq(sh_xy_at(p, u, v, i, j, k))) +
                                        (sq(sh_xy_at(p, u, v, i - 1, j, k)) + sq(sh_xy_at(p, u, v, i, j - 1, k))));
        shear = sqrt(sh_xx_sq + sh_xy_sq);
    }
    if (p.leith_Kh) {   // vert_vort_mag = grad_vort_mag_h (+ 0: no modified Leith)
        const double gx = 0.5 * (vort_dx_at(p, u, v, i, j, k) + vort_dx_at(p, u, v, i, j - 1, k));
        const double gy = 0.5 * (vort_dy_at(p, u, v, i, j, k) + vort_dy_at(p, u, v, i - 1, j, k));
        vvm = sqrt(sq(gx) + sq(gy)) + 0.0;
    }
    if (p.bound) hrat = hrat_at(p, h, i, j, k);
    double rem = 1.0, Kh = 0.0;
    if (p.laplacian) {
        Kh = p.Kh;
        if (p.smag_Kh) Kh = fmax(Kh, 0.15 * 0.15 * a2 * shear);
        if (p.leith_Kh) Kh = fmax(Kh, 1.0 * (sqrt(a2) * a2) * vvm * HV_INV_PI3);
        Kh = fmax(Kh, 0.0);
        if (p.bound) {   // better_bound_Kh and better_bound_Ah together
            const double Kh_max_here = hrat * (0.25 * a2 / 1.0);
            if (Kh >= Kh_max_here) {
                rem = 0.0;
                Kh = Kh_max_here;
            } else if (Kh > 0.0) {
                rem = 1.0 - Kh / Kh_max_here;
            }
        }
    }
    *Kh_out = Kh;
    if (!p.biharmonic) return;
    double Ah = p.Ah;
    if (p.smag_Ah) Ah = fmax(Ah, 0.06 * 0.06 * (a2 * a2) * shear);
    if (p.leith_Ah) {
        const double Del2vort_h = 0.25 * ((del2vort_q_at(p, u, v, i, j, k) + del2vort_q_at(p, u, v, i - 1, j - 1, k)) +
                                          (del2vort_q_at(p, u, v, i - 1, j, k) + del2vort_q_at(p, u, v, i, j - 1, k)));
        const double h3 = sqrt(a2) * a2;
        Ah = fmax(Ah, 1.0 * h3 * h3 * fabs(Del2vort_h) * HV_INV_PI6);
    }
    if (p.bound) Ah = fmin(Ah, rem * hrat * (0.0625 * (a2 * a2) / 1.0));
    *Ah_out = Ah;
}

// Kh (which = 0) or Ah (1) at a q point of Isq..Ieq x Jsq..Jeq (:897-1023)
__device__ inline double visc_q_point(const HV &p, const double *u, const double *v, const double *h, int I, int J,
                                      int k, int which)
{
    const Dims &d = p.d;
    const double a2 = p.areaT[IX2(d, I, J)];
    const bool smag = which == 0 ? p.smag_Kh : p.smag_Ah;
    const bool leith = which == 0 ? p.leith_Kh : p.leith_Ah;
    double x = which == 0 ? p.Kh : p.Ah;
    if (smag) {
        const double sh_xx_sq = 0.25 * ((sq(sh_xx_at(p, u, v, I, J, k)) + sq(sh_xx_at(p, u, v, I + 1, J + 1, k))) +
                                        (sq(sh_xx_at(p, u, v, I + 1, J, k)) + sq(sh_xx_at(p, u, v, I, J + 1, k))));
        const double sh_xy_sq = sq(sh_xy_at(p, u, v, I, J, k));
        x = fmax(x, (which == 0 ? 0.15 * 0.15 * a2 : 0.06 * 0.06 * (a2 * a2)) * sqrt(sh_xx_sq + sh_xy_sq));
    }
    if (leith) {
        const double h3 = sqrt(a2) * a2;
        if (which == 0) {
            const double gx = 0.5 * (vort_dx_at(p, u, v, I, J, k) + vort_dx_at(p, u, v, I + 1, J, k));
            const double gy = 0.5 * (vort_dy_at(p, u, v, I, J, k) + vort_dy_at(p, u, v, I, J + 1, k));
            x = fmax(x, 1.0 * h3 * sqrt(sq(gx) + sq(gy)) * HV_INV_PI3);
        } else {
            x = fmax(x, 1.0 * h3 * h3 * fabs(del2vort_q_at(p, u, v, I, J, k)) * HV_INV_PI6);
        }
    }
    if (which == 0) x = fmax(x, 0.0);   // Kh_bg_min
    if (p.bound) {
        const double h_min = 0.25 * ((hrat_at(p, h, I, J, k) + hrat_at(p, h, I + 1, J + 1, k)) +
                                     (hrat_at(p, h, I + 1, J, k) + hrat_at(p, h, I, J + 1, k)));
        x = fmin(x, h_min * (which == 0 ? 0.25 * a2 / 1.0 : 0.0625 * (a2 * a2) / 1.0));
    }
    return x;
}

// Kh and Ah seen by the stress at h point (i, j) of Isq..Ieq+1 x Jsq..Jeq+1
__device__ inline void visc_seen(const HV &p, const double *u, const double *v, const double *h, int i, int j, int k,
                                 double *Kh, double *Ah)
{
    const Dims &d = p.d;
    if (interior(d, i, j)) {
        visc_h_point(p, u, v, h, i, j, k, Kh, Ah);
    } else if (q_range(d, i, j)) {
        if (k > 1) {
            *Kh = p.laplacian ? visc_q_point(p, u, v, h, i, j, k - 1, 0) : 0.0;
            *Ah = p.biharmonic ? visc_q_point(p, u, v, h, i, j, k - 1, 1) : 0.0;
        } else {
            *Kh = p.ring_Kh[IX2(d, i, j)];
            *Ah = p.ring_Ah[IX2(d, i, j)];
        }
    } else {
        *Kh = 0.0;
        *Ah = 0.0;
    }
}

__device__ inline double str_xx_x(const HV &p, const double *u, const double *v, const double *h, int i, int j, int k)
{
    const Dims &d = p.d;
    double Kh = 0.0, Ah = 0.0;
    visc_seen(p, u, v, h, i, j, k, &Kh, &Ah);
    double str = p.laplacian ? -(Kh * sh_xx_at(p, u, v, i, j, k)) : 0.0;
    if (p.biharmonic) {
        const double d_del2u = (p.IdyCu[IX2(d, i, j)] * p.Del2u[IX3(d, i, j, k)]) -
                               (p.IdyCu[IX2(d, i - 1, j)] * p.Del2u[IX3(d, i - 1, j, k)]);
        const double d_del2v = (p.IdxCv[IX2(d, i, j)] * p.Del2v[IX3(d, i, j, k)]) -
                               (p.IdxCv[IX2(d, i, j - 1)] * p.Del2v[IX3(d, i, j - 1, k)]);
        str = str + Ah * ((p.DY_dxT[IX2(d, i, j)] * d_del2u) - (p.DX_dyT[IX2(d, i, j)] * d_del2v));
    }
    return str * (h[IX3(d, i, j, k)] * p.reduction_xx[IX2(d, i, j)]);
}

__device__ inline double str_xy_x(const HV &p, const double *u, const double *v, const double *h, int I, int J, int k)
{
    const Dims &d = p.d;
    const long long c2 = IX2(d, I, J);
    double str = p.laplacian ? -(visc_q_point(p, u, v, h, I, J, k, 0) * sh_xy_at(p, u, v, I, J, k)) : 0.0;
    if (p.biharmonic) {
        const double d_str =
            visc_q_point(p, u, v, h, I, J, k, 1) *
            ((p.DY_dxBu[c2] * ((p.Del2v[IX3(d, I + 1, J, k)] * p.IdyCv[IX2(d, I + 1, J)]) -
                               (p.Del2v[IX3(d, I, J, k)] * p.IdyCv[c2]))) +
             (p.DX_dyBu[c2] * ((p.Del2u[IX3(d, I, J + 1, k)] * p.IdxCu[IX2(d, I, J + 1)]) -
                               (p.Del2u[IX3(d, I, J, k)] * p.IdxCu[c2]))));
        str = str + d_str;
    }
    const double hq = 0.25 * ((h[IX3(d, I, J, k)] + h[IX3(d, I + 1, J + 1, k)]) +
                              (h[IX3(d, I + 1, J, k)] + h[IX3(d, I, J + 1, k)]));
    if (p.no_slip) return str * (hq * p.reduction_xy[c2]);
    return str * (hq * p.mask2dBu[c2] * p.reduction_xy[c2]);
}

// diffu, diffv with the closures (the same ranges and expressions as k_hv_main)
__global__ void __launch_bounds__(64) k_hv_closures(HV p, const double *__restrict__ u, const double *__restrict__ v,
                                                    const double *__restrict__ h, double *__restrict__ diffu,
                                                    double *__restrict__ diffv)
{
    const Dims &d = p.d;
    const int i = d.isd + blockIdx.x * blockDim.x + threadIdx.x;
    const int j = d.jsd + blockIdx.y;
    const int k = 1 + blockIdx.z;
    if (i > d.ied) return;
    const long long c = IX3(d, i, j, k), c2 = IX2(d, i, j);
    double du = 0.0, dv = 0.0;
    if (i >= d.isc - 1 && i <= d.iec && j >= d.jsc && j <= d.jec) {
        du = ((p.IdxCu[c2] * ((p.dx2q[IX2(d, i, j - 1)] * str_xy_x(p, u, v, h, i, j - 1, k)) -
                              (p.dx2q[c2] * str_xy_x(p, u, v, h, i, j, k))) +
               p.IdyCu[c2] * ((p.dy2h[c2] * str_xx_x(p, u, v, h, i, j, k)) -
                              (p.dy2h[IX2(d, i + 1, j)] * str_xx_x(p, u, v, h, i + 1, j, k)))) *
              p.IareaCu[c2]) / (h_u_at(p, h, i, j, k) + p.h_neglect);
    }
    if (i >= d.isc && i <= d.iec && j >= d.jsc - 1 && j <= d.jec) {
        dv = ((p.IdyCv[c2] * ((p.dy2q[IX2(d, i - 1, j)] * str_xy_x(p, u, v, h, i - 1, j, k)) -
                              (p.dy2q[c2] * str_xy_x(p, u, v, h, i, j, k))) -
               p.IdxCv[c2] * ((p.dx2h[c2] * str_xx_x(p, u, v, h, i, j, k)) -
                              (p.dx2h[IX2(d, i, j + 1)] * str_xx_x(p, u, v, h, i, j + 1, k)))) *
              p.IareaCv[c2]) / (h_v_at(p, h, i, j, k) + p.h_neglect);
    }
    diffu[c] = du;
    diffv[c] = dv;
}

// After a call: the q-point Kh and Ah of its last layer at the ring points
// (is-1, js-1..je) and (is..ie, js-1), for the next call's first layer
__global__ void k_hv_keep_ring(HV p, const double *__restrict__ u, const double *__restrict__ v,
                               const double *__restrict__ h)
{
    const Dims &d = p.d;
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    const int ncol = d.jec - d.jsc + 2, nrow = d.iec - d.isc + 1;
    if (q >= ncol + nrow) return;
    const int I = q < ncol ? d.isc - 1 : d.isc + (q - ncol);
    const int J = q < ncol ? d.jsc - 1 + q : d.jsc - 1;
    p.ring_Kh[IX2(d, I, J)] = p.laplacian ? visc_q_point(p, u, v, h, I, J, d.nk, 0) : 0.0;
    p.ring_Ah[IX2(d, I, J)] = p.biharmonic ? visc_q_point(p, u, v, h, I, J, d.nk, 1) : 0.0;
}

// ---------------------------------------------------------------------------
// Grids whose metric arrays are constant (over is-2..ie+2 x js-2..je+2, every
// point the stencil reads): every operator -- constant Kh and Ah, Smagorinsky,
// Leith, the bounds -- as one march, as the fused momentum stencil does it.  A
// wave holds 64 columns of one layer and walks along j: i neighbours by lane
// shifts, j neighbours kept from the rows before, so each strain, vorticity and
// its derivatives, thickness ratio, viscosity, Del2 and stress is formed once per
// point.  At step r row r arrives; suffix 0 marks its h points, 1 the q and h
// points of row r - 1, and so on.  The expressions are the general kernels' with
// the constant metric values, so the results are bit-identical to theirs.
//
// The stress at the h points of the ring (is-1 or js-1) reads Kh and Ah of the
// previous layer's q points: k_hv_ring forms those for every layer beforehand
// (a few thousand points), and the march loads them with the row.
//
// What bounds it: VALU issue with the closures, memory without.  360x283x50 with
// Smagorinsky, the bounds and the biharmonic term: 116 us per call (march 98, ring
// 11) against 3240 us when one thread per point evaluated every work value it
// needed from u, v and h (and Del2 in a launch of its own, 214 us of them).
// Laplacian, against the 64 x 8 tile staged in LDS that it replaces: 28x20x7 8 us
// (18), 300x260x25 20 (38), 471x363x50 83 (94), 500x500x75 178 (180), 720x720x75 346
// (379), 1440x1440x20 381 (392).  With FP64 masks and five rows walked beyond a chunk
// it was slower than the tile from 500x500 on (199, 395 and 436 us): memory bounds it.
// With the biharmonic term it saves the Del2 launch and arrays: 720x720x75 374 (2600).
template <bool SMAG, bool LEITH, bool BOUND, bool BIH>
struct HVMarch {
    static constexpr bool CL = SMAG || LEITH || BOUND;
    static constexpr int LM = CL || BIH ? 2 : 1;                       // lanes that only lend, west
    static constexpr int RM = LEITH ? 3 : CL || BIH ? 2 : 1;           // and east
    static constexpr int OUT = 64 - LM - RM;
    // rows read before the first and after the last row written
    static constexpr int BEFORE = CL || BIH ? 2 : 1, AFTER = CL ? 3 : BIH ? 2 : 1;
};

// compact index of a ring point: (is-1, js-1..je), then (is..ie, js-1)
__device__ inline int ring_index(const Dims &d, int I, int J)
{
    return I == d.isc - 1 ? J - (d.jsc - 1) : d.jec - d.jsc + 2 + (I - d.isc);
}
__host__ __device__ inline int ring_points(const Dims &d)
{
    return (d.jec - d.jsc + 2) + (d.iec - d.isc + 1);
}

// Kh (ring_q[0 ..]) and Ah (ring_q[nk*points ..]) of every layer at the ring points
__global__ void __launch_bounds__(64) k_hv_ring(HV p, const double *__restrict__ u, const double *__restrict__ v,
                                                const double *__restrict__ h, double *__restrict__ ring_q)
{
    const Dims &d = p.d;
    const int q = blockIdx.x * 64 + threadIdx.x, n = ring_points(d), k = 1 + blockIdx.y;
    if (q >= n) return;
    const int ncol = d.jec - d.jsc + 2;
    const int I = q < ncol ? d.isc - 1 : d.isc + (q - ncol);
    const int J = q < ncol ? d.jsc - 1 + q : d.jsc - 1;
    ring_q[(long long)(k - 1) * n + q] = p.laplacian ? visc_q_point(p, u, v, h, I, J, k, 0) : 0.0;
    ring_q[(long long)(d.nk + k - 1) * n + q] = p.biharmonic ? visc_q_point(p, u, v, h, I, J, k, 1) : 0.0;
}

// After the call: the last layer's, for the next call's first layer
__global__ void __launch_bounds__(64) k_hv_keep_last(HV p, const double *__restrict__ ring_q)
{
    const Dims &d = p.d;
    const int q = blockIdx.x * 64 + threadIdx.x, n = ring_points(d);
    if (q >= n) return;
    const int ncol = d.jec - d.jsc + 2;
    const long long c = IX2(d, q < ncol ? d.isc - 1 : d.isc + (q - ncol), q < ncol ? d.jsc - 1 + q : d.jsc - 1);
    p.ring_Kh[c] = ring_q[(long long)(d.nk - 1) * n + q];
    p.ring_Ah[c] = ring_q[(long long)(2 * d.nk - 1) * n + q];
}

// BITS: the masks from one byte per point (the constant-coefficient operators on
// 0/1 masks: their FP64 planes, read again in every layer, were 0.6 of the 1.74 GB
// a call read at 720x720x75)
template <bool SMAG, bool LEITH, bool BOUND, bool BIH, bool BITS>
__global__ void __launch_bounds__(256) k_hv_march(HV p, HVUniform g, const double *__restrict__ u,
                                                  const double *__restrict__ v, const double *__restrict__ h,
                                                  const double *__restrict__ ring_q, double *__restrict__ diffu,
                                                  double *__restrict__ diffv, int strips, int chunks, int rows)
{
    using M = HVMarch<SMAG, LEITH, BOUND, BIH>;
    const Dims &d = p.d;
    const int is = d.isc, ie = d.iec, js = d.jsc, je = d.jec;
    const int t = xcd_tile(blockIdx.x, gridDim.x) * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int per = strips * chunks, k = t / per + 1, tq = t % per, strip = tq % strips;
    if (k > d.nk) return;
    const int ja = d.jsd + (tq / strips) * rows, jb = ja + rows - 1 < d.jed ? ja + rows - 1 : d.jed;
    const int lane = threadIdx.x & 63;
    const int i = d.isd + strip * M::OUT - M::LM + lane;
    const unsigned col = (unsigned)((i < d.isd ? d.isd : i > d.ied ? d.ied : i) - d.isd);   // clamped: such lanes only lend
    const bool mine = lane >= M::LM && lane < 64 - M::RM && i <= d.ied;
    const bool in_i = i >= is && i <= ie, in_I = i >= is - 1 && i <= ie;
    const long long n1 = d.n1, layer = (long long)(k - 1) * d.s2;
    auto row_of = [&](int j) -> long long { return (long long)((j < d.jsd ? d.jsd : j > d.jed ? d.jed : j) - d.jsd) * n1; };
    auto in_j = [&](int j) { return j >= js && j <= je; };       // h rows
    auto in_J = [&](int j) { return j >= js - 1 && j <= je; };   // q rows
    // the ring's viscosities: of the previous layer (the first layer: of the
    // previous call), or the constants (zero in the first layer of the first call)
    const bool ring_strip = strip * M::OUT - M::LM + d.isd <= is - 1;
    const int nring = ring_points(d);
    const double ring_c = k == 1 && p.first_call ? 0.0 : 1.0;
    const double Kh_c = ring_c * p.Kh, Ah_c = ring_c * p.Ah;
    const double area = g.areaT, h3 = sqrt(area) * area;
    const bool lap = p.laplacian;
    const double smag_K = p.smag_Kh ? 0.15 * 0.15 * area : 0.0, smag_A = 0.06 * 0.06 * (area * area);

    double nu, nv, nh, nmT = 0.0, nmB = 0.0, nrK = 0.0, nrA = 0.0;   // the newest row, in flight until its step
    unsigned nm = 0;
    auto load = [&](int r) __attribute__((always_inline)) {
        const long long row = row_of(r), o = layer + row;
        nu = (u + o)[col];
        nv = (v + o)[col];
        nh = (h + o)[col];
        if (BITS) {
            nm = (p.mask_bits + row)[col];
        } else {
            nmT = (p.mask2dT + row)[col];
            nmB = (p.mask2dBu + row)[col];
        }
        if (M::CL) {   // the ring's Kh and Ah for the stress of h row r - 2
            const int J = r - 2;
            if (in_J(J) && (ring_strip || J == js - 1)) {
                const bool on = i == is - 1 || (J == js - 1 && in_i);
                if (on) {
                    const int q = ring_index(d, i, J);
                    if (k > 1) {
                        nrK = ring_q[(long long)(k - 2) * nring + q];
                        nrA = ring_q[(long long)(d.nk + k - 2) * nring + q];
                    } else {
                        nrK = p.ring_Kh[IX2(d, i, J)];
                        nrA = p.ring_Ah[IX2(d, i, J)];
                    }
                }
            }
        }
    };
    double u1, v1, ve1, h1, he1, mh1, mB1;                                     // row r - 1
    double xx1 = 0.0, xx1e = 0.0, xx2 = 0.0, xy2 = 0.0, hq2 = 0.0, h2 = 0.0, hu2 = 0.0, hv2 = 0.0, hv3 = 0.0, mB2 = 0.0;
    double sxx1 = 0.0, sxx1e = 0.0, sxy2 = 0.0, sxy2w = 0.0, shear_h2 = 0.0, shear_q2 = 0.0;      // SMAG
    double vort2 = 0.0, vdx2 = 0.0, vdy2 = 0.0, vvm2 = 0.0, d2v3_ = 0.0;                          // LEITH (d2v3_: row r - 3)
    double hrat2 = 1.0;                                                                           // BOUND
    double d2u2 = 0.0, d2v2 = 0.0, d2v3 = 0.0;                                                    // BIH
    double tx3 = 0.0, ty3 = 0.0;                                               // stresses of row r - 3
    auto mask_T = [&]() { return BITS ? (double)(nm & 1u) : nmT; };
    auto mask_B = [&]() { return BITS ? (double)((nm >> 1) & 1u) : nmB; };
    load(ja - M::BEFORE);
    u1 = nu; v1 = nv; h1 = nh; ve1 = east(nv); he1 = east(nh); mh1 = mask_T() * nh; mB1 = mask_B();
    load(ja - M::BEFORE + 1);
    for (int r = ja - M::BEFORE + 1; r <= jb + 3; ++r) {
        const double u0 = nu, v0 = nv, h0 = nh, mT0 = mask_T(), mB0 = mask_B(), rK = nrK, rA = nrA;
        if (r < jb + M::AFTER) load(r + 1);   // later rows reach no output
        const double ve0 = east(v0), he0 = east(h0), mh0 = mT0 * h0;
        // tension at the h points of row r (:503-530)
        const double dudx = g.DY_dxT * ((g.IdyCu * u0) - (g.IdyCu * west(u0)));
        const double dvdy = g.DX_dyT * ((g.IdxCv * v0) - (g.IdxCv * v1));
        const double xx0 = dudx - dvdy, xx0e = east(xx0);
        // row r - 1: shearing strain (:513-547), thicknesses (:551-562)
        const double dvdx = g.DY_dxBu * ((ve1 * g.IdyCv) - (v1 * g.IdyCv));
        const double dudy = g.DX_dyBu * ((u0 * g.IdxCu) - (u1 * g.IdxCu));
        const double slip = p.no_slip ? (2.0 - mB1) : mB1;
        const double xy1 = slip * (dvdx + dudy);
        const double hq1 = 0.25 * ((h1 + he0) + (he1 + h0));
        const double hu1 = 0.5 * (mh1 + east(mh1)), hv1 = 0.5 * (mh1 + mh0);
        const bool in1 = in_i && in_j(r - 1), in2 = in_i && in_j(r - 2);
        double hrat1 = 1.0;
        if (BOUND) {   // hrat_min (:730-737)
            const double h_min = fmin(fmin(fmin(hu1, west(hu1)), hv1), hv2);
            const double x = fmin(1.0, h_min / (h1 + p.h_neglect));
            hrat1 = in1 ? x : 1.0;
        }
        double sxx0 = 0.0, sxx0e = 0.0, sxy1 = 0.0, sxy1w = 0.0, shear_h1 = 0.0, shear_q1 = 0.0;
        if (SMAG) {    // Shear_mag at h (:710-720) and q points
            sxx0 = sq(xx0); sxx0e = east(sxx0);
            sxy1 = sq(xy1); sxy1w = west(sxy1);
            shear_h1 = sqrt(sxx1 + 0.25 * ((sxy2w + sxy1) + (sxy1w + sxy2)));
            shear_q1 = sqrt(0.25 * ((sxx1 + sxx0e) + (sxx1e + sxx0)) + sxy1);
        }
        double vort1 = 0.0, vdx1 = 0.0, vdy1 = 0.0, vvm1 = 0.0, d2_2 = 0.0, d2h2 = 0.0, gq2 = 0.0;
        if (LEITH) {   // vorticity (:612-626), its gradients (:629-645) and Laplacian (:648-659)
            vort1 = slip * (dvdx - dudy);
            const double vx = g.DY_dxBu_v * ((vort1 * g.IdyCu) - (west(vort1) * g.IdyCu));
            const double vy = g.DX_dyBu_v * ((vort1 * g.IdxCv) - (vort2 * g.IdxCv));
            vdx1 = in1 ? vx : 0.0;
            vdy1 = in_I && in_j(r - 1) ? vy : 0.0;
            vvm1 = sqrt(sq(0.5 * (vdx1 + vdx2)) + sq(0.5 * (vdy1 + west(vdy1)))) + 0.0;
            const double vdx2e = east(vdx2);
            gq2 = sqrt(sq(0.5 * (vdx2 + vdx2e)) + sq(0.5 * (vdy2 + vdy1)));
            const double x = g.DY_dxBu * ((vdx2e * g.IdyCv) - (vdx2 * g.IdyCv)) +
                             g.DX_dyBu * ((vdy1 * g.IdxCu) - (vdy2 * g.IdxCu));
            d2_2 = in_I && in_J(r - 2) ? x : 0.0;
            d2h2 = 0.25 * ((d2_2 + west(d2v3_)) + (west(d2_2) + d2v3_));
        }
        double d2u1 = 0.0, d2v1 = 0.0;
        if (BIH) {     // Del2u, Del2v of row r - 1 (:587-607), zero outside their ranges
            const double x = g.Idx2dyCu * ((g.dx2q * xy1) - (g.dx2q * xy2)) +
                             g.Idxdy2u * ((g.dy2h * xx1e) - (g.dy2h * xx1));
            const double y = g.Idxdy2v * ((g.dy2q * xy1) - (g.dy2q * west(xy1))) -
                             g.Idx2dyCv * ((g.dx2h * xx0) - (g.dx2h * xx1));
            d2u1 = in_I && in_j(r - 1) ? x : 0.0;
            d2v1 = in_i && in_J(r - 1) ? y : 0.0;
        }
        // row r - 2: viscosities at h (:743-863) and q points (:897-1023)
        double Kh = p.Kh, Ah = p.Ah, Kq = p.Kh, Aq = p.Ah;
        if (M::CL) {
            double rem = 1.0;
            const double Kh_top = hrat2 * (0.25 * area / 1.0), Ah_top = 0.0625 * (area * area) / 1.0;
            if (SMAG && p.smag_Kh) {
                Kh = fmax(Kh, smag_K * shear_h2);
                Kq = fmax(Kq, smag_K * shear_q2);
            }
            if (LEITH) {
                Kh = fmax(Kh, 1.0 * h3 * vvm2 * HV_INV_PI3);
                Kq = fmax(Kq, 1.0 * h3 * gq2 * HV_INV_PI3);
            }
            Kh = fmax(Kh, 0.0);
            Kq = fmax(Kq, 0.0);
            double hmin_q = 1.0;
            if (BOUND) {
                hmin_q = 0.25 * ((hrat2 + east(hrat1)) + (east(hrat2) + hrat1));
                if (lap) {
                    const double part = 1.0 - Kh / Kh_top;
                    rem = Kh >= Kh_top ? 0.0 : (Kh > 0.0 ? part : 1.0);
                    Kh = Kh >= Kh_top ? Kh_top : Kh;
                }
                Kq = fmin(Kq, hmin_q * (0.25 * area / 1.0));
            }
            if (BIH) {
                if (SMAG) {
                    Ah = fmax(Ah, smag_A * shear_h2);
                    Aq = fmax(Aq, smag_A * shear_q2);
                }
                if (LEITH) {
                    Ah = fmax(Ah, 1.0 * h3 * h3 * fabs(d2h2) * HV_INV_PI6);
                    Aq = fmax(Aq, 1.0 * h3 * h3 * fabs(d2_2) * HV_INV_PI6);
                }
                if (BOUND) {
                    Ah = fmin(Ah, rem * hrat2 * Ah_top);
                    Aq = fmin(Aq, hmin_q * Ah_top);
                }
            }
        }
        const bool ring2 = in_I && in_J(r - 2);   // and not in2
        Kh = in2 ? Kh : (ring2 ? (M::CL ? rK : Kh_c) : 0.0);
        if (BIH) Ah = in2 ? Ah : (ring2 ? (M::CL ? rA : Ah_c) : 0.0);
        // its stresses times thickness (:807-895, :954-1053)
        double tx2 = lap ? -(Kh * xx2) : 0.0, ty2 = lap ? -(Kq * xy2) : 0.0;
        if (BIH) {
            const double d_del2u = (g.IdyCu * d2u2) - (g.IdyCu * west(d2u2));
            const double d_del2v = (g.IdxCv * d2v2) - (g.IdxCv * d2v3);
            tx2 = tx2 + Ah * ((g.DY_dxT * d_del2u) - (g.DX_dyT * d_del2v));
            ty2 = ty2 + Aq * ((g.DY_dxBu * ((east(d2v2) * g.IdyCv) - (d2v2 * g.IdyCv))) +
                              (g.DX_dyBu * ((d2u1 * g.IdxCu) - (d2u2 * g.IdxCu))));
        }
        tx2 = tx2 * (h2 * g.red_xx);
        ty2 = p.no_slip ? ty2 * (hq2 * g.red_xy) : ty2 * (hq2 * mB2 * g.red_xy);
        // diffu of row r - 2 and diffv of row r - 3 (:1059-1078), zero outside their ranges
        const double tx2e = east(tx2), ty3w = west(ty3);
        if (r - 2 >= ja && r - 2 <= jb) {
            const double x = ((g.IdxCu * ((g.dx2q * ty3) - (g.dx2q * ty2)) + g.IdyCu * ((g.dy2h * tx2) - (g.dy2h * tx2e))) *
                              g.IareaCu) / (hu2 + p.h_neglect);
            if (mine) (diffu + layer + row_of(r - 2))[col] = in_I && in_j(r - 2) ? x : 0.0;
        }
        if (r - 3 >= ja) {
            const double x = ((g.IdyCv * ((g.dy2q * ty3w) - (g.dy2q * ty3)) - g.IdxCv * ((g.dx2h * tx3) - (g.dx2h * tx2))) *
                              g.IareaCv) / (hv3 + p.h_neglect);
            if (mine) (diffv + layer + row_of(r - 3))[col] = in_i && in_J(r - 3) ? x : 0.0;
        }
        tx3 = tx2; ty3 = ty2;
        hv3 = hv2; hv2 = hv1; hu2 = hu1; hq2 = hq1; h2 = h1; mB2 = mB1;
        xx2 = xx1; xx1 = xx0; xx1e = xx0e; xy2 = xy1;
        if (SMAG) { sxx1 = sxx0; sxx1e = sxx0e; sxy2 = sxy1; sxy2w = sxy1w; shear_h2 = shear_h1; shear_q2 = shear_q1; }
        if (LEITH) { vort2 = vort1; vdx2 = vdx1; vdy2 = vdy1; vvm2 = vvm1; d2v3_ = d2_2; }
        if (BOUND) hrat2 = hrat1;
        if (BIH) { d2v3 = d2v2; d2u2 = d2u1; d2v2 = d2v1; }
        u1 = u0; v1 = v0; ve1 = ve0; h1 = h0; he1 = he0; mh1 = mh0; mB1 = mB0;
    }
}

static HV make_hv(const mom6h_hor_visc_cs *cs)
{
    HV p;
    p.d = cs->d;
    p.Kh = cs->Kh; p.Ah = cs->Ah; p.h_neglect = cs->h_neglect;
    p.laplacian = cs->laplacian; p.biharmonic = cs->biharmonic; p.no_slip = cs->no_slip;
    p.first_call = cs->calls == 0;
    p.DY_dxT = cs->DY_dxT; p.DX_dyT = cs->DX_dyT; p.DY_dxBu = cs->DY_dxBu; p.DX_dyBu = cs->DX_dyBu;
    p.IdyCu = cs->IdyCu; p.IdxCu = cs->IdxCu; p.IdyCv = cs->IdyCv; p.IdxCv = cs->IdxCv;
    p.IareaCu = cs->IareaCu; p.IareaCv = cs->IareaCv; p.mask2dT = cs->mask2dT; p.mask2dBu = cs->mask2dBu;
    p.reduction_xx = cs->reduction_xx; p.reduction_xy = cs->reduction_xy;
    p.dy2h = cs->dy2h; p.dx2h = cs->dx2h; p.dy2q = cs->dy2q; p.dx2q = cs->dx2q;
    p.Idx2dyCu = cs->Idx2dyCu; p.Idxdy2u = cs->Idxdy2u; p.Idx2dyCv = cs->Idx2dyCv; p.Idxdy2v = cs->Idxdy2v;
    p.mask_bits = cs->mask_bits;
    p.Del2u = cs->Del2u; p.Del2v = cs->Del2v;
    p.smag_Kh = cs->smagorinsky && cs->laplacian;
    p.smag_Ah = cs->smagorinsky && cs->biharmonic;
    p.leith_Kh = cs->leith;
    p.leith_Ah = cs->leith && cs->biharmonic;
    p.bound = cs->better_bound;
    p.areaT = cs->areaT; p.dxBu = cs->dxBu; p.dyBu = cs->dyBu; p.IdxBu = cs->IdxBu; p.IdyBu = cs->IdyBu;
    p.ring_Kh = cs->ring_Kh; p.ring_Ah = cs->ring_Ah;
    return p;
}

static bool closures_on(const mom6h_hor_visc_cs *cs) { return cs->smagorinsky || cs->leith || cs->better_bound; }

// every metric that the options in use read is constant
static bool march_takes(const mom6h_hor_visc_cs *cs)
{
    return cs->uniform && (!cs->biharmonic || cs->bih_uniform) && (!closures_on(cs) || cs->area_uniform) &&
           (!cs->leith || cs->leith_uniform);
}

int hor_visc_scratch(mom6h_hor_visc_cs *cs)
{
    if (!cs->biharmonic || (march_takes(cs) && !cs->general)) return MOM6H_OK;
    const size_t n3 = (size_t)cs->d.s2 * cs->d.nk;
    int rc = cs->Del2u ? MOM6H_OK : dev_alloc(&cs->Del2u, n3, true);
    if (!rc && !cs->Del2v) rc = dev_alloc(&cs->Del2v, n3, true);
    return rc;
}

// the march's launch over the data domain: chunks of rows that leave about
// four waves per SIMD, at least 8, at most 48 with the closures (a chunk then walks
// five rows more than it writes) and 40 without (Laplacian, us per call at 32 / 40 /
// 48 / 56 / 64: 500x500x75 179 / 178 / 185 / 175 / 184, 720x720x75 347 / 346 / 355 /
// 358 / 362, 1440x1440x20 377 / 381 / 391 / 394 / 388)
template <bool SMAG, bool LEITH, bool BOUND, bool BIH>
static void launch_march(const mom6h_hor_visc_cs *cs, const HV &p, const double *u, const double *v, const double *h,
                         double *diffu, double *diffv, hipStream_t s)
{
    const Dims &d = cs->d;
    constexpr int OUT = HVMarch<SMAG, LEITH, BOUND, BIH>::OUT;
    const int strips = (d.n1 + OUT - 1) / OUT;
    int rows = (int)std::min(HVMarch<SMAG, LEITH, BOUND, BIH>::CL ? 48LL : 40LL, std::max(8LL, (long long)strips * d.n2 * d.nk / 4096));
    int chunks = (d.n2 + rows - 1) / rows;
    rows = (d.n2 + chunks - 1) / chunks;
    chunks = (d.n2 + rows - 1) / rows;
    const long long tasks = (long long)strips * chunks * d.nk;
    const unsigned blocks = (unsigned)((tasks + 3) / 4);
    constexpr bool CL = HVMarch<SMAG, LEITH, BOUND, BIH>::CL;
    if (!CL && cs->mask_bits)
        k_hv_march<SMAG, LEITH, BOUND, BIH, !CL><<<blocks, 256, 0, s>>>(p, cs->g, u, v, h, cs->ring_q, diffu, diffv,
                                                                      strips, chunks, rows);
    else
        k_hv_march<SMAG, LEITH, BOUND, BIH, false><<<blocks, 256, 0, s>>>(p, cs->g, u, v, h, cs->ring_q, diffu, diffv,
                                                                        strips, chunks, rows);
}

template <bool SMAG, bool LEITH, bool BOUND>
static void launch_march(const mom6h_hor_visc_cs *cs, const HV &p, const double *u, const double *v, const double *h,
                         double *diffu, double *diffv, hipStream_t s)
{
    if (cs->biharmonic) launch_march<SMAG, LEITH, BOUND, true>(cs, p, u, v, h, diffu, diffv, s);
    else launch_march<SMAG, LEITH, BOUND, false>(cs, p, u, v, h, diffu, diffv, s);
}

template <bool SMAG>
static void launch_march(const mom6h_hor_visc_cs *cs, const HV &p, const double *u, const double *v, const double *h,
                         double *diffu, double *diffv, hipStream_t s)
{
    if (cs->leith) {
        if (cs->better_bound) launch_march<SMAG, true, true>(cs, p, u, v, h, diffu, diffv, s);
        else launch_march<SMAG, true, false>(cs, p, u, v, h, diffu, diffv, s);
    } else {
        if (cs->better_bound) launch_march<SMAG, false, true>(cs, p, u, v, h, diffu, diffv, s);
        else launch_march<SMAG, false, false>(cs, p, u, v, h, diffu, diffv, s);
    }
}

// every metric the stencil reads constant over is-2..ie+2 x js-2..je+2
static bool hv_uniform(const Dims &d, std::initializer_list<std::pair<const double *, double *>> fields)
{
    for (const auto &f : fields)
        if (!uniform_over(d, f.first, d.isc - 2, d.iec + 2, d.jsc - 2, d.jec + 2, f.second)) return false;
    return true;
}

}  // namespace mom6h

using namespace mom6h;

extern "C" {

int mom6h_hor_visc_init(mom6h_hor_visc_cs **out, int isd, int ied, int jsd, int jed, int isc,
                        int iec, int jsc, int jec, int nz, double Kh, double h_neglect,
                        const double *DY_dxT, const double *DX_dyT, const double *DY_dxBu,
                        const double *DX_dyBu, const double *IdyCu, const double *IdxCu,
                        const double *IdyCv, const double *IdxCv, const double *IareaCu,
                        const double *IareaCv, const double *mask2dT, const double *mask2dBu,
                        const double *reduction_xx, const double *reduction_xy, const double *dy2h,
                        const double *dx2h, const double *dy2q, const double *dx2q)
{
    MOM6H_REQUIRE(out != nullptr, "mom6h_hor_visc_init: NULL cs");
    MOM6H_REQUIRE(isd < isc - 1 && iec + 1 < ied && jsd < jsc - 1 && jec + 1 < jed && isc <= iec &&
                      jsc <= jec && nz >= 1,
                  "mom6h_hor_visc_init: needs two halo cells on every side");
    MOM6H_REQUIRE(DY_dxT && DX_dyT && DY_dxBu && DX_dyBu && IdyCu && IdxCu && IdyCv && IdxCv &&
                      IareaCu && IareaCv && mask2dT && mask2dBu && reduction_xx && reduction_xy &&
                      dy2h && dx2h && dy2q && dx2q,
                  "mom6h_hor_visc_init: NULL metric");
    auto *cs = new mom6h_hor_visc_cs();
    cs->d = make_dims(isd, ied, jsd, jed, isc, iec, jsc, jec, nz);
    cs->Kh = Kh;
    cs->Ah = 0.0;
    cs->h_neglect = h_neglect;
    cs->laplacian = 1;
    cs->biharmonic = 0;
    cs->no_slip = 0;
    cs->calls = 0;
    const size_t n2 = (size_t)cs->d.s2;
    int rc = 0;
    const double *src[] = {DY_dxT, DX_dyT, DY_dxBu, DX_dyBu, IdyCu, IdxCu, IdyCv, IdxCv, IareaCu,
                           IareaCv, mask2dT, mask2dBu, reduction_xx, reduction_xy, dy2h, dx2h, dy2q, dx2q};
    double **dst[] = {&cs->DY_dxT, &cs->DX_dyT, &cs->DY_dxBu, &cs->DX_dyBu, &cs->IdyCu, &cs->IdxCu,
                      &cs->IdyCv, &cs->IdxCv, &cs->IareaCu, &cs->IareaCv, &cs->mask2dT, &cs->mask2dBu,
                      &cs->reduction_xx, &cs->reduction_xy, &cs->dy2h, &cs->dx2h, &cs->dy2q, &cs->dx2q};
    for (size_t q = 0; q < sizeof(src) / sizeof(src[0]); ++q) rc = rc ? rc : dev_upload(dst[q], src[q], n2);
    if (rc) {
        mom6h_hor_visc_end(cs);
        return rc;
    }
    HVUniform &g = cs->g;
    cs->uniform = hv_uniform(cs->d, {{DY_dxT, &g.DY_dxT}, {DX_dyT, &g.DX_dyT}, {DY_dxBu, &g.DY_dxBu},
                                     {DX_dyBu, &g.DX_dyBu}, {IdyCu, &g.IdyCu}, {IdxCu, &g.IdxCu},
                                     {IdyCv, &g.IdyCv}, {IdxCv, &g.IdxCv}, {IareaCu, &g.IareaCu},
                                     {IareaCv, &g.IareaCv}, {reduction_xx, &g.red_xx},
                                     {reduction_xy, &g.red_xy}, {dy2h, &g.dy2h}, {dx2h, &g.dx2h},
                                     {dy2q, &g.dy2q}, {dx2q, &g.dx2q}});
    if (cs->uniform && binary_mask(mask2dT, n2) && binary_mask(mask2dBu, n2)) {
        rc = dev_alloc_bytes((void **)&cs->mask_bits, n2, false);
        if (!rc) rc = launch_mask_bits(MaskJobs{1, {{cs->mask2dT, cs->mask2dBu, cs->mask_bits, (long long)n2}}}, nullptr);
        if (!rc && hipStreamSynchronize(nullptr) != hipSuccess) rc = set_error(MOM6H_ESTATE, "mask conversion failed");
        if (rc) {
            mom6h_hor_visc_end(cs);
            return rc;
        }
    }
    *out = cs;
    return MOM6H_OK;
}

int mom6h_hor_visc_set_options(mom6h_hor_visc_cs *cs, int laplacian, int biharmonic, double Ah,
                               int no_slip, const double *Idx2dyCu, const double *Idxdy2u,
                               const double *Idx2dyCv, const double *Idxdy2v)
{
    MOM6H_REQUIRE(cs != nullptr, "mom6h_hor_visc_set_options: NULL cs");
    MOM6H_REQUIRE(!biharmonic || (Idx2dyCu && Idxdy2u && Idx2dyCv && Idxdy2v),
                  "mom6h_hor_visc_set_options: biharmonic needs its four metrics");
    if (biharmonic && !cs->biharmonic) {
        const size_t n2 = (size_t)cs->d.s2;
        int rc = 0;
        rc = rc ? rc : dev_upload(&cs->Idx2dyCu, Idx2dyCu, n2);
        rc = rc ? rc : dev_upload(&cs->Idxdy2u, Idxdy2u, n2);
        rc = rc ? rc : dev_upload(&cs->Idx2dyCv, Idx2dyCv, n2);
        rc = rc ? rc : dev_upload(&cs->Idxdy2v, Idxdy2v, n2);
        if (rc) return rc;
        HVUniform &g = cs->g;
        cs->bih_uniform = hv_uniform(cs->d, {{Idx2dyCu, &g.Idx2dyCu}, {Idxdy2u, &g.Idxdy2u},
                                             {Idx2dyCv, &g.Idx2dyCv}, {Idxdy2v, &g.Idxdy2v}});
    }
    const int was = cs->biharmonic;
    cs->biharmonic = biharmonic;
    const int rc = hor_visc_scratch(cs);
    if (rc) {
        cs->biharmonic = was;   // never on without its work fields
        return rc;
    }
    cs->laplacian = laplacian;
    cs->no_slip = no_slip;
    cs->Ah = Ah;
    return MOM6H_OK;
}

int mom6h_hor_visc(mom6h_hor_visc_cs *cs, const double *u, const double *v, const double *h,
                   double *diffu, double *diffv, void *stream)
{
    MOM6H_REQUIRE(cs != nullptr, "mom6h_hor_visc: NULL cs");
    MOM6H_REQUIRE(u && v && h && diffu && diffv, "mom6h_hor_visc: NULL array");
    const Dims &d = cs->d;
    hipStream_t s = (hipStream_t)stream;
    HV p = make_hv(cs);
    if (march_takes(cs) && !cs->general) {
        const unsigned nring = (unsigned)((ring_points(d) + 63) / 64);
        if (closures_on(cs)) {
            k_hv_ring<<<dim3(nring, d.nk), 64, 0, s>>>(p, u, v, h, cs->ring_q);
            MOM6H_LAUNCH_CHECK();
        }
        if (cs->smagorinsky) launch_march<true>(cs, p, u, v, h, diffu, diffv, s);
        else launch_march<false>(cs, p, u, v, h, diffu, diffv, s);
        MOM6H_LAUNCH_CHECK();
        if (closures_on(cs)) {
            k_hv_keep_last<<<nring, 64, 0, s>>>(p, cs->ring_q);
            MOM6H_LAUNCH_CHECK();
        }
        cs->calls++;
        return MOM6H_OK;
    }
    if (cs->biharmonic) {
        const int ni = d.iec - (d.isc - 1) + 1, nj = d.jec - (d.jsc - 1) + 1;
        dim3 b(64), g((ni + 63) / 64, nj, d.nk);
        k_hv_del2<<<g, b, 0, s>>>(p, u, v);
        MOM6H_LAUNCH_CHECK();
    }
    dim3 b(64), g((d.n1 + 63) / 64, d.n2, d.nk);
    if (closures_on(cs)) {
        k_hv_closures<<<g, b, 0, s>>>(p, u, v, h, diffu, diffv);
        MOM6H_LAUNCH_CHECK();
        k_hv_keep_ring<<<(ring_points(d) + 63) / 64, 64, 0, s>>>(p, u, v, h);
    } else {
        k_hv_main<<<g, b, 0, s>>>(p, u, v, h, diffu, diffv);
    }
    MOM6H_LAUNCH_CHECK();
    cs->calls++;
    return MOM6H_OK;
}

int mom6h_hor_visc_set_closures(mom6h_hor_visc_cs *cs, int smagorinsky, int leith, int better_bound,
                                const double *areaT, const double *dxBu, const double *dyBu, const double *IdxBu,
                                const double *IdyBu)
{
    MOM6H_REQUIRE(cs != nullptr, "mom6h_hor_visc_set_closures: NULL cs");
    MOM6H_REQUIRE(cs->calls == 0, "mom6h_hor_visc_set_closures: before the first mom6h_hor_visc call");
    MOM6H_REQUIRE(!(smagorinsky || leith || better_bound) || areaT, "mom6h_hor_visc_set_closures: needs areaT");
    MOM6H_REQUIRE(!leith || (dxBu && dyBu && IdxBu && IdyBu), "mom6h_hor_visc_set_closures: Leith needs the q-point metrics");
    const size_t n2 = (size_t)cs->d.s2;
    int rc = 0;
    // the metrics are the first call's; the march's values are taken with them
    HVUniform &g = cs->g;
    if (smagorinsky || leith || better_bound) {
        if (!cs->areaT) {
            rc = dev_upload(&cs->areaT, areaT, n2);
            cs->area_uniform = hv_uniform(cs->d, {{areaT, &g.areaT}});
        }
        if (!rc && !cs->ring_Kh) rc = dev_alloc(&cs->ring_Kh, n2, true);
        if (!rc && !cs->ring_Ah) rc = dev_alloc(&cs->ring_Ah, n2, true);
        if (!rc && !cs->ring_q) rc = dev_alloc(&cs->ring_q, (size_t)2 * cs->d.nk * ring_points(cs->d), false);
    }
    if (!rc && leith && !cs->dxBu) {
        rc = dev_upload(&cs->dxBu, dxBu, n2);
        rc = rc ? rc : dev_upload(&cs->dyBu, dyBu, n2);
        rc = rc ? rc : dev_upload(&cs->IdxBu, IdxBu, n2);
        rc = rc ? rc : dev_upload(&cs->IdyBu, IdyBu, n2);
        double dx = 0.0, dy = 0.0, idx = 0.0, idy = 0.0;
        cs->leith_uniform = hv_uniform(cs->d, {{dxBu, &dx}, {dyBu, &dy}, {IdxBu, &idx}, {IdyBu, &idy}});
        g.DY_dxBu_v = dy * idx;
        g.DX_dyBu_v = dx * idy;
    }
    if (rc) return rc;
    const int was[3] = {cs->smagorinsky, cs->leith, cs->better_bound};
    cs->smagorinsky = smagorinsky;
    cs->leith = leith;
    cs->better_bound = better_bound;
    rc = hor_visc_scratch(cs);
    if (rc) {
        cs->smagorinsky = was[0];
        cs->leith = was[1];
        cs->better_bound = was[2];
    }
    return rc;
}

int mom6h_hor_visc_end(mom6h_hor_visc_cs *cs)
{
    if (!cs) return MOM6H_OK;
    for (double *p : {cs->DY_dxT, cs->DX_dyT, cs->DY_dxBu, cs->DX_dyBu, cs->IdyCu, cs->IdxCu,
                      cs->IdyCv, cs->IdxCv, cs->IareaCu, cs->IareaCv, cs->mask2dT, cs->mask2dBu,
                      cs->reduction_xx, cs->reduction_xy, cs->dy2h, cs->dx2h, cs->dy2q, cs->dx2q,
                      cs->Idx2dyCu, cs->Idxdy2u, cs->Idx2dyCv, cs->Idxdy2v, cs->Del2u, cs->Del2v,
                      cs->areaT, cs->dxBu, cs->dyBu, cs->IdxBu, cs->IdyBu, cs->ring_Kh, cs->ring_Ah, cs->ring_q})
        dev_free(p);
    if (cs->mask_bits) (void)hipFree(cs->mask_bits);
    delete cs;
    return MOM6H_OK;
}

}  // extern "C"
