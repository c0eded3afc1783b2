// mom6h_fused.h -- kernels of the fused step for grids with uniform metrics.
#pragma once
#include <functional>
#include <string>

#include "mom6h_internal.h"

namespace mom6h {

// One value per metric array (the arrays of a uniform grid are constant; the
// values are read from the arrays, so every expression sees the same numbers
// as the general kernels do).
struct UMetrics {
    double areaT, IareaT, dxT, IdxT, dyCu, dy_Cu, dxCu, IdxCu, IdyCu, dxCv, dyCv, IdxCv, IdyCv;
    double IareaBu, IareaCu, IareaCv, Area_q;
    double DY_dxT, DX_dyT, DY_dxBu, DX_dyBu, dx2h, dy2h, dx2q, dy2q;
    double Idx2dyCu, Idxdy2u, Idx2dyCv, Idxdy2v;   // biharmonic (hor_visc_init :262-283)
};

// The metric values in the stencil's arithmetic type (T = double: unchanged)
template <typename T>
struct UMetT {
    T areaT, IareaT, dxT, IdxT, dyCu, dy_Cu, dxCu, IdxCu, IdyCu, dxCv, dyCv, IdxCv, IdyCv;
    T IareaBu, IareaCu, IareaCv, Area_q;
    T DY_dxT, DX_dyT, DY_dxBu, DX_dyBu, dx2h, dy2h, dx2q, dy2q;
    T Idx2dyCu, Idxdy2u, Idx2dyCv, Idxdy2v;
    __host__ __device__ explicit UMetT(const UMetrics &g)
        : areaT((T)g.areaT), IareaT((T)g.IareaT), dxT((T)g.dxT), IdxT((T)g.IdxT), dyCu((T)g.dyCu),
          dy_Cu((T)g.dy_Cu), dxCu((T)g.dxCu), IdxCu((T)g.IdxCu), IdyCu((T)g.IdyCu), dxCv((T)g.dxCv),
          dyCv((T)g.dyCv), IdxCv((T)g.IdxCv), IdyCv((T)g.IdyCv), IareaBu((T)g.IareaBu), IareaCu((T)g.IareaCu),
          IareaCv((T)g.IareaCv), Area_q((T)g.Area_q), DY_dxT((T)g.DY_dxT), DX_dyT((T)g.DX_dyT),
          DY_dxBu((T)g.DY_dxBu), DX_dyBu((T)g.DX_dyBu), dx2h((T)g.dx2h), dy2h((T)g.dy2h), dx2q((T)g.dx2q),
          dy2q((T)g.dy2q), Idx2dyCu((T)g.Idx2dyCu), Idxdy2u((T)g.Idxdy2u), Idx2dyCv((T)g.Idx2dyCv),
          Idxdy2v((T)g.Idxdy2v)
    {
    }
};

// Arguments of the fused momentum stencil.  T is the type of the 3D layer
// fields and of the stencil arithmetic (double: the reference's FP64; float:
// the mixed-precision form); Coriolis stays FP64 in memory.
template <typename T>
struct MomArgsT {
    Dims d;
    UMetrics g;
    T Kh, h_neglect, fdt;
    int no_slip;
    const T *u, *v, *h;               // stencil inputs
    const T *bu, *bv;                 // bases of the update (may alias ou/ov)
    T *ou, *ov;
    const unsigned char *mask;        // the 0/1 masks per point: bit 0 mask2dT, bit 1 mask2dBu
    const double *CoriolisBu;         // constant along every row
    T Ah;
    int bih;                          // biharmonic viscosity beside the Laplacian (Ah)
    int march;                        // rows a wave marches through (0: chosen from the grid)
};
using MomArgs = MomArgsT<double>;

// One grid, or every member of an ensemble in one launch (d_args: the members'
// arguments on the device, h_args: the same on the host, their march set by
// plan_momentum_batch: `rows`, or with 0 chosen from all members' grids)
template <typename T>
int launch_momentum(const MomArgsT<T> &a, hipStream_t s);
template <typename T>
int plan_momentum_batch(MomArgsT<T> *h_args, int n, int rows);
template <typename T>
int launch_momentum_batch(const MomArgsT<T> *d_args, const MomArgsT<T> *h_args, int n, hipStream_t s);

// Del2u and Del2v of the biharmonic term as fields, for a caller that asks for
// them (the stencil itself keeps them in registers)
template <typename T>
struct Del2Args {
    Dims d;
    UMetrics g;
    int no_slip;
    const T *u, *v;
    const double *mask2dBu;
    T *del2u, *del2v;   // written on their own ranges only, zero elsewhere from allocation
};
template <typename T>
int launch_del2(const Del2Args<T> &a, hipStream_t s);

// MomArgsT::mask from the FP64 masks (2D, n points each) of one or several grids
struct MaskJob {
    const double *mask2dT, *mask2dBu;
    unsigned char *bits;
    long long n;
};
struct MaskJobs {
    int n;
    MaskJob j[kMaxMembers];
};
int launch_mask_bits(const MaskJobs &jobs, hipStream_t s);

// Rows a wave of the momentum stencil marches through for the options
// momentum_tile and momentum_splits (0 while neither is set: chosen from the grid)
inline int march_rows(int tile, int splits)
{
    if (!tile && !splits) return 0;
    const int rows = 8 * (tile ? tile : 8) / (splits ? splits : 1);
    return rows < 4 ? 4 : rows;
}

// Chooses the options momentum_tile and momentum_splits by timing launch (what a
// step does with the stencil) on stream s under each candidate, which set puts in
// force: marches of 64 to 4 rows and the one chosen from the grid (0, 0), which
// stays unless another is faster by more than 1%.  After a warm-up one round over the
// candidates, then up to `reps` in all over those within 5% of the best, in
// alternating order; the shortest time of each counts.  Leaves the choice set and
// adds the times to the report.
int tune_march(hipStream_t s, int reps, const std::function<int(int tile, int splits)> &set,
               const std::function<int()> &launch, std::string *report);

// true and the common value when every element of a[0..n) is identical
inline bool uniform_value(const double *a, size_t n, double *v)
{
    for (size_t q = 1; q < n; ++q)
        if (!(a[q] == a[0])) return false;
    *v = a[0];
    return true;
}

// true when every element of a[0..n) is 0 or 1 (a land/sea mask the fused
// momentum stencil can read as a bit)
inline bool binary_mask(const double *a, size_t n)
{
    for (size_t q0 = 0; q0 < n; q0 += 4096) {   // whole blocks without a branch: vector compares
        const size_t q1 = q0 + 4096 < n ? q0 + 4096 : n;
        bool ok = true;
        for (size_t q = q0; q < q1; ++q) ok &= (a[q] == 0.0) | (a[q] == 1.0);
        if (!ok) return false;
    }
    return true;
}

// true when the 2D field a (ni x nj, i fastest) is constant along every row
// j (f-plane and beta-plane Coriolis: the fused momentum stencil reads one
// value per row)
inline bool rows_uniform(const double *a, size_t ni, size_t nj)
{
    for (size_t j = 0; j < nj; ++j)
        for (size_t i = 1; i < ni; ++i)
            if (!(a[j * ni + i] == a[j * ni])) return false;
    return true;
}

}  // namespace mom6h
