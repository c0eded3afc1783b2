// mom6h_fused.hip -- fused momentum stencil for grids with uniform metrics.
//
// One launch performs, for every layer, what the reference does in four
// module calls (app/rk2_serial_driver.F90:236-270 and :316-350):
//   compute_transports (:544-561) -> hor_visc (src/serial/mom6_hor_visc_serial.F90,
//   Laplacian, with or without the biharmonic term) -> CorAdCalc
//   (src/serial/mom6_coriolis_serial.F90, Sadourny energy scheme) -> velocity
//   update  ou = base + fdt*(CA + diff)
// The transports, tendencies, strains, Del2 fields and potential vorticity
// never leave the registers (the march below).
//
// On a uniform grid every metric array holds one value; the kernels take those
// values (read from the arrays at set-up) and keep the reference's operation
// order, so the results are bit-identical to the general kernels.  The
// Kh/Ah ring of hor_visc and the never-written hArea rows of CorAdCalc only
// matter for diffu/diffv/CAu/CAv outside the velocity-update ranges; inside
// them the q values on row js-1 and column is-1 still see the zero hArea the
// reference reads, exactly as here.
#include <algorithm>
#include <cstdio>

#include "mom6h_fused.h"

namespace mom6h {

// Division in the stencil's type: exact in FP64 (the reference's arithmetic);
// in the FP32 form a product with the hardware reciprocal (about 1 ulp, the
// rounding scale of the FP32 stencil itself)
template <typename T>
__device__ __forceinline__ T sdiv(T num, T den)
{
    if constexpr (sizeof(T) == 4) return num * __builtin_amdgcn_rcpf(den);
    else return num / den;
}

// One wave marches along j through rows ja..jb of one layer, lane l holding
// column i0 + l: the i neighbours come from the neighbouring lanes (DPP), the
// j neighbours are the values kept from the rows before.  So every strain, q,
// KE, transport and stress is formed once per point, no LDS, no barrier and no
// index arithmetic beyond a row pointer; the outermost LM lanes on either side
// only lend their values (the next strip's wave computes them).  At step r the
// row r arrives (its loads were issued a step before); the h-point terms of
// row r and the q-point terms of row p = r - 1 follow, and with them the
// outputs of row p.  BIH: Del2u and Del2v of row p come next, then the stresses
// of h row p and q row p - 1, and the outputs are those of row p - 1 (its
// Coriolis terms kept for one step).
//
// What bounds it: 225 VALU instructions per row of 62 points (FP64, Laplacian)
// against the 370 of a 64 x 8 tile staged in LDS with its recomputed ring, 38
// KB of LDS and two barriers per layer, which was VALU-bound.  At 720x720x75
// predictor and corrector now take 0.84 ms together at 16 rows (1.30 ms before):
// 1.69 and 2.32 GB of memory traffic at 4.8 TB/s, near the 5.4 of a plain copy, with
// the VALU 87% and 81% busy: both about equal.  FP32: 0.44 ms (0.68), VALU issue; with
// the biharmonic term 0.53 ms, which took 1.40 ms with Del2 formed by a launch of its
// own and read back.
template <typename T, bool BIH>
struct March {
    static constexpr int LM = BIH ? 2 : 1;          // lent lanes on either side
    static constexpr int OUT = 64 - 2 * LM;         // columns a wave updates
    static constexpr int LAG = BIH ? 2 : 1;         // rows between the newest row and the outputs
};

// SAME: the base of the update is the stencil's own input (the predictor), so
// its row is at hand; otherwise (the corrector) it is loaded
template <typename T, bool BIH, bool SAME>
__device__ __forceinline__ void march(const MomArgsT<T> &a, int strip, int ja, int jb, int k)
{
    using M = March<T, BIH>;
    const Dims &d = a.d;
    const UMetT<T> g(a.g);
    const int is = d.isc, ie = d.iec, js = d.jsc, je = d.jec;
    const int lane = threadIdx.x & 63;
    const int i = is + strip * M::OUT - M::LM + lane;
    const unsigned col = (unsigned)((i <= d.ied ? i : d.ied) - d.isd);   // clamped: such lanes only lend
    const bool mine = lane >= M::LM && lane < 64 - M::LM;
    const bool out_u = mine && i <= ie - 1, out_v = mine && i <= ie;
    const bool west_edge = i < is;
    const bool del2u_col = i >= is - 1 && i <= ie, del2v_col = i >= is && i <= ie;
    const long long n1 = d.n1, layer = (long long)(k - 1) * d.s2;
    const T slip_a = a.no_slip ? T(2.0) : T(0.0), slip_b = a.no_slip ? T(-1.0) : T(1.0);

    // the newest row (in flight until its step)
    T nu, nv, nh, ncor, nbu = T(0.0), nbv = T(0.0);
    unsigned nm;
    auto load = [&](int r) __attribute__((always_inline)) {
        const long long row = (long long)(r - d.jsd) * n1, o = layer + row;
        nu = (a.u + o)[col];
        nv = (a.v + o)[col];
        nh = (a.h + o)[col];
        nm = (a.mask + row)[col];
        ncor = (T)a.CoriolisBu[row];   // constant along the row
        if (!SAME) {                   // the base of the row that step r finishes
            const int b = r - M::LAG;
            if (b >= ja) {
                const long long ob = layer + (long long)(b - d.jsd) * n1;
                nbu = (a.bu + ob)[col];
                nbv = (a.bv + ob)[col];
            }
        }
    };

    // kept from the row before (p): state, masked thickness, h-point terms
    T u_p, v_p, ve_p, h_p, he_p, mh_p, mBu_p, cor_p, hAu_p;
    T KE_p = T(0.0), KEe_p = T(0.0), uh_p = T(0.0), uhw_p = T(0.0);
    T sxx_p = T(0.0), sxxe_p = T(0.0);              // stress*h (BIH: the strain sh_xx)
    // kept from q row p - 1
    T q_s = T(0.0), vhs_s = T(0.0), sxy_s = T(0.0); // (BIH: sxy_s is the strain sh_xy)
    // BIH: kept for the outputs of row p - 1
    T CAu_o = T(0.0), CAv_o = T(0.0), hu_o = T(1.0), hv_o = T(1.0), hqm_s = T(0.0), h_o = T(0.0);
    T d2u_s = T(0.0), d2v_s = T(0.0);               // Del2 of row p - 1
    T txx_o = T(0.0), txxe_o = T(0.0), txy_o = T(0.0);   // stress*h of h row p - 1, stress*hq of q row p - 2
    T u_o = T(0.0), v_o = T(0.0);                   // SAME: the base of row p - 1

    const int r0 = ja - M::LAG;
    load(r0);
    {
        u_p = nu; v_p = nv; h_p = nh;
        ve_p = east(nv); he_p = east(nh);
        mh_p = (T)(nm & 1u) * nh;
        mBu_p = (T)((nm >> 1) & 1u);
        cor_p = ncor;
        // never formed on row js-1 (mom6_coriolis_serial.F90:142-152): zero
        hAu_p = r0 < js ? T(0.0) : T(0.5) * ((g.areaT * h_p) + (g.areaT * he_p));
    }
    load(r0 + 1);
    for (int r = r0 + 1; r <= jb + M::LAG; ++r) {
        const T u = nu, v = nv, h = nh, cor = ncor, bu = nbu, bv = nbv;
        const T mT = (T)(nm & 1u), mBu = (T)((nm >> 1) & 1u);
        if (r < jb + M::LAG) load(r + 1);
        const int p = r - 1;
        const T uw = west(u), ve = east(v), he = east(h);
        const T mh = mT * h;
        // h points of row r: strain and KE (mom6_hor_visc_serial.F90:503-510,
        // mom6_coriolis_serial.F90:196-203), transport uh
        const T dudx = g.DY_dxT * ((g.IdyCu * u) - (g.IdyCu * uw));
        const T dvdy = g.DX_dyT * ((g.IdxCv * v) - (g.IdxCv * v_p));
        const T sh_xx = dudx - dvdy;
        const T KE = sdiv(T(0.25) * ((g.dyCu * (u * u) + g.dyCu * (uw * uw)) +
                                     (g.dxCv * (v * v) + g.dxCv * (v_p * v_p))), g.areaT);
        const T KEe = east(KE);
        const T uh = u * T(0.5) * (h + he) * g.dyCu;
        const T uhw = west(uh);
        // q points of row p: potential vorticity (:134-168), transport vh
        const T hAu = T(0.5) * ((g.areaT * h) + (g.areaT * he));
        const T hAv = T(0.5) * ((g.areaT * h_p) + (g.areaT * h));
        const T hAve = T(0.5) * ((g.areaT * he_p) + (g.areaT * he));
        const T rel_vort = mBu_p * (((ve_p * g.dyCv) - (v_p * g.dyCv)) - ((u * g.dxCu) - (u_p * g.dxCu))) * g.IareaBu;
        const T hArea_q = (hAu_p + hAu) + ((west_edge ? T(0.0) : hAv) + hAve);
        const T q = (cor_p + rel_vort) * sdiv(g.Area_q, hArea_q + T(1.0e-20));
        const T qw = west(q);
        const T vh = v_p * T(0.5) * (h_p + h) * g.dxCv;
        const T vhs = east(vh) + vh;
        // CAu and CAv of row p, Sadourny (:208-226)
        const T CAu = T(0.25) * ((q * vhs) + (q_s * vhs_s)) * g.IdxCu - (KEe_p - KE_p) * g.IdxCu;
        const T CAv = -(T(0.25) * ((qw * (uhw_p + uhw)) + (q * (uh_p + uh))) * g.IdyCv) - (KE - KE_p) * g.IdyCv;
        // strain at the q points of row p (:513-547) and the thickness there
        const T dvdx = g.DY_dxBu * ((ve_p * g.IdyCv) - (v_p * g.IdyCv));
        const T dudy = g.DX_dyBu * ((u * g.IdxCu) - (u_p * g.IdxCu));
        const T sh_xy = (slip_a + slip_b * mBu_p) * (dvdx + dudy);
        const T hq = T(0.25) * ((h_p + he) + (he_p + h));
        const T hqm = hq * (a.no_slip ? T(1.0) : mBu_p);
        const T h_u = T(0.5) * (mh_p + east(mh_p)) + a.h_neglect, h_v = T(0.5) * (mh_p + mh) + a.h_neglect;

        // outputs of row jo (diffu :1059-1067, diffv :1070-1078, velocity
        // update): stresses xx of its h points (own and east) and of the row
        // above, xy of its q points (own and west) and of the row below
        auto finish = [&](int jo, T Cu, T Cv, T den_u, T den_v, T xx, T xxe, T xx_n, T xy, T xy_s, T b_u, T b_v)
                          __attribute__((always_inline)) {
            const T xyw = west(xy);
            if (jo < ja) return;
            const T diffu = sdiv((g.IdxCu * ((g.dx2q * xy_s) - (g.dx2q * xy)) +
                                  g.IdyCu * ((g.dy2h * xx) - (g.dy2h * xxe))) * g.IareaCu, den_u);
            const T diffv = sdiv((g.IdyCv * ((g.dy2q * xyw) - (g.dy2q * xy)) -
                                  g.IdxCv * ((g.dx2h * xx) - (g.dx2h * xx_n))) * g.IareaCv, den_v);
            const long long o = layer + (long long)(jo - d.jsd) * n1;
            if (out_u) (a.ou + o)[col] = b_u + a.fdt * (Cu + diffu);
            if (out_v && jo <= je - 1) (a.ov + o)[col] = b_v + a.fdt * (Cv + diffv);
        };
        if constexpr (!BIH) {
            const T xx = -(a.Kh * sh_xx) * h, xxe = east(xx);
            const T xy = -(a.Kh * sh_xy) * hqm;
            finish(p, CAu, CAv, h_u, h_v, sxx_p, sxxe_p, xx, xy, sxy_s, SAME ? u_p : bu, SAME ? v_p : bv);
            sxx_p = xx; sxxe_p = xxe;
            sxy_s = xy;
        } else {
            // Del2u on u points I = is-1..ie, j = js..je and Del2v on v points
            // i = is..ie, J = js-1..je of row p (:587-607), zero elsewhere
            const T sh_xxe = east(sh_xx);
            T d2u = g.Idx2dyCu * ((g.dx2q * sh_xy) - (g.dx2q * sxy_s)) +
                    g.Idxdy2u * ((g.dy2h * sxxe_p) - (g.dy2h * sxx_p));
            T d2v = g.Idxdy2v * ((g.dy2q * sh_xy) - (g.dy2q * west(sh_xy))) -
                    g.Idx2dyCv * ((g.dx2h * sh_xx) - (g.dx2h * sxx_p));
            if (!(del2u_col && p >= js && p <= je)) d2u = T(0.0);
            if (!(del2v_col && p >= js - 1 && p <= je)) d2v = T(0.0);
            // stress*h at the h points of row p (:824-886)
            const T d_del2u = (g.IdyCu * d2u) - (g.IdyCu * west(d2u));
            const T d_del2v = (g.IdxCv * d2v) - (g.IdxCv * d2v_s);
            const T txx = (-(a.Kh * sxx_p) + a.Ah * ((g.DY_dxT * d_del2u) - (g.DX_dyT * d_del2v))) * h_p;
            const T txxe = east(txx);
            // stress*hq at the q points of row p - 1 (:979-1036)
            const T txy = (-(a.Kh * sxy_s) +
                           a.Ah * ((g.DY_dxBu * ((east(d2v_s) * g.IdyCv) - (d2v_s * g.IdyCv))) +
                                   (g.DX_dyBu * ((d2u * g.IdxCu) - (d2u_s * g.IdxCu))))) * hqm_s;
            finish(p - 1, CAu_o, CAv_o, hu_o, hv_o, txx_o, txxe_o, txx, txy, txy_o, SAME ? u_o : bu, SAME ? v_o : bv);
            CAu_o = CAu; CAv_o = CAv; hu_o = h_u; hv_o = h_v; hqm_s = hqm;
            txx_o = txx; txxe_o = txxe; txy_o = txy;
            d2u_s = d2u; d2v_s = d2v;
            sxx_p = sh_xx; sxxe_p = sh_xxe;
            sxy_s = sh_xy;
            u_o = u_p; v_o = v_p;
        }
        q_s = q; vhs_s = vhs;
        u_p = u; v_p = v; ve_p = ve; h_p = h; he_p = he; mh_p = mh; mBu_p = mBu; cor_p = cor;
        hAu_p = r < js ? T(0.0) : hAu;
        KE_p = KE; KEe_p = KEe; uh_p = uh; uhw_p = uhw;
    }
}

// Tasks of one grid: strips (fastest), row chunks of `rows` rows, layers; one
// wave per task, four waves per block
struct MarchPlan {
    int strips, chunks, rows;
    long long tasks;
};

inline MarchPlan march_plan(const Dims &d, bool bih, int rows)
{
    MarchPlan m;
    const int out = bih ? March<double, true>::OUT : March<double, false>::OUT, nj = d.jec - d.jsc + 1;
    m.strips = (d.iec - d.isc + out) / out;
    m.chunks = (nj + rows - 1) / rows;
    m.rows = (nj + m.chunks - 1) / m.chunks;   // even chunks
    m.chunks = (nj + m.rows - 1) / m.rows;
    m.tasks = (long long)m.strips * m.chunks * d.nk;
    return m;
}

template <typename T, bool BIH, bool SAME>
__device__ __forceinline__ void march_task(const MomArgsT<T> &a, int strips, int chunks, int rows, int block)
{
    const int t = block * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int per = strips * chunks, k = t / per, q = t % per;
    if (k >= a.d.nk) return;
    const int ja = a.d.jsc + (q / strips) * rows, jb = ja + rows - 1 < a.d.jec ? ja + rows - 1 : a.d.jec;
    march<T, BIH, SAME>(a, q % strips, ja, jb, k + 1);
}

template <typename T, bool BIH, bool SAME>
__global__ void __launch_bounds__(256) k_momentum(MomArgsT<T> a, int strips, int chunks, int rows)
{
    march_task<T, BIH, SAME>(a, strips, chunks, rows, xcd_tile(blockIdx.x, gridDim.x));
}

// every member of an ensemble in one launch, renumbered per XCD over the whole
// batch; mp.nbx, mp.nby: strips and chunks, a.march the rows of a chunk
template <typename T, bool BIH, bool SAME>
__global__ void __launch_bounds__(256) k_momentum_batch(const MomArgsT<T> *__restrict__ args, BatchMap mp)
{
    int m, local;
    batch_locate(mp, xcd_tile(blockIdx.x, gridDim.x), m, local);
    const MomArgsT<T> a = args[m];
    march_task<T, BIH, SAME>(a, mp.nbx[m], mp.nby[m], a.march, local);
}

template <typename T, bool BIH, bool SAME>
void march_launch(const MomArgsT<T> &a, const MarchPlan &m, hipStream_t s)
{
    k_momentum<T, BIH, SAME><<<(unsigned)((m.tasks + 3) / 4), 256, 0, s>>>(a, m.strips, m.chunks, m.rows);
}

// Rows of a march when the caller sets none: a long march repeats less (each
// starts LAG rows early and walks LAG rows beyond its last), a short one gives more
// waves.  Four waves per SIMD (4096) are worth shorter marches, down to 4 rows;
// beyond that 32 rows serve every size within 4%.  us per step (predictor and
// corrector, among a step's other kernels) at 128 / 64 / 32 / 16 / 8 / 4 rows, FP64:
// 140x100x40: 185 / 99 / 71 / 43 / 33 / 28; 180x180x75: 174 / 124 / 84 / 67 / 63 /
// 65; 720x720x75: 955 / 879 / 860 / 841 / 851 / 909; 1440x1440x75: 3288 / 3150 /
// 3128 / 3089 / 3179 / 3562; FP32 720x720x75: 564 / 487 / 456 / 443 / 465 / 526, with
// the biharmonic term 627 / 533 / 530 / 546 / 611 / 759.
constexpr long long kMarchWaves = 4096;
inline int auto_rows(long long wave_rows)
{
    return (int)std::min(32LL, std::max(4LL, wave_rows / kMarchWaves));
}
inline long long wave_rows(const Dims &d, bool bih)
{
    return march_plan(d, bih, 1).tasks;
}

template <typename T>
int launch_momentum(const MomArgsT<T> &a, hipStream_t s)
{
    const bool same = a.u == a.bu && a.v == a.bv;
    const MarchPlan m = march_plan(a.d, a.bih, a.march > 0 ? a.march : auto_rows(wave_rows(a.d, a.bih)));
    if (a.bih) {
        if (same) march_launch<T, true, true>(a, m, s);
        else march_launch<T, true, false>(a, m, s);
    } else {
        if (same) march_launch<T, false, true>(a, m, s);
        else march_launch<T, false, false>(a, m, s);
    }
    MOM6H_LAUNCH_CHECK();
    return MOM6H_OK;
}

template <typename T>
int plan_momentum_batch(MomArgsT<T> *h_args, int n, int rows)
{
    MOM6H_REQUIRE(n >= 1 && n <= kMaxMembers, "momentum batch: 1..%d members", kMaxMembers);
    if (rows <= 0) {
        long long all = 0;
        for (int m = 0; m < n; ++m) all += wave_rows(h_args[m].d, h_args[m].bih);
        rows = auto_rows(all);
    }
    for (int m = 0; m < n; ++m) h_args[m].march = march_plan(h_args[m].d, h_args[m].bih, rows).rows;
    return MOM6H_OK;
}

template <typename T>
int launch_momentum_batch(const MomArgsT<T> *d_args, const MomArgsT<T> *h_args, int n, hipStream_t s)
{
    MOM6H_REQUIRE(n >= 1 && n <= kMaxMembers, "momentum batch: 1..%d members", kMaxMembers);
    const bool bih = h_args[0].bih, same = h_args[0].u == h_args[0].bu && h_args[0].v == h_args[0].bv;
    BatchMap mp{};
    mp.n = n;
    for (int m = 0; m < n; ++m) {
        const MomArgsT<T> &a = h_args[m];
        MOM6H_REQUIRE((a.bih != 0) == bih, "momentum batch: members differ in biharmonic");
        MOM6H_REQUIRE((a.u == a.bu && a.v == a.bv) == same, "momentum batch: members differ in their base fields");
        MOM6H_REQUIRE(a.march >= 1, "momentum batch: members have no march plan");
        const MarchPlan p = march_plan(a.d, bih, a.march);
        MOM6H_REQUIRE(p.rows == a.march, "momentum batch: a member's march plan is not its launch's");
        mp.nbx[m] = p.strips;
        mp.nby[m] = p.chunks;
        mp.first[m + 1] = mp.first[m] + (int)((p.tasks + 3) / 4);
    }
    const unsigned nb = (unsigned)mp.first[n];
    if (bih) {
        if (same) k_momentum_batch<T, true, true><<<nb, 256, 0, s>>>(d_args, mp);
        else k_momentum_batch<T, true, false><<<nb, 256, 0, s>>>(d_args, mp);
    } else {
        if (same) k_momentum_batch<T, false, true><<<nb, 256, 0, s>>>(d_args, mp);
        else k_momentum_batch<T, false, false><<<nb, 256, 0, s>>>(d_args, mp);
    }
    MOM6H_LAUNCH_CHECK();
    return MOM6H_OK;
}

// One timing of each candidate in a fixed order, predictor only, chose 128 rows at
// 720x720x75 (0.42 ms, in the first place after a pause) where a step's two
// launches then took 1.01 ms, against 0.89 ms with 16 rows: the clock moves for
// some milliseconds after a pause, and the corrector's extra base rows weigh on long
// marches.  Hence the warm-up, the alternating order and both phases: 20 ms with reps
// = 3 there.
int tune_march(hipStream_t s, int reps, const std::function<int(int, int)> &set, const std::function<int()> &launch,
               std::string *report)
{
    constexpr int N = 6;
    const int tile[N] = {0, 8, 4, 4, 4, 4}, splits[N] = {0, 1, 1, 2, 4, 8};   // auto, 64 .. 4 rows
    hipEvent_t a = nullptr, b = nullptr;
    int rc = hipEventCreate(&a) == hipSuccess && hipEventCreate(&b) == hipSuccess
                 ? MOM6H_OK
                 : set_error(MOM6H_ENOMEM, "event creation failed");
    // ms per launch of candidate q, over n launches
    auto time = [&](int q, int n) -> float {
        float t = 0.f;
        if (!rc) rc = set(tile[q], splits[q]);
        if (!rc && hipEventRecord(a, s) != hipSuccess) rc = set_error(MOM6H_ESTATE, "event record failed");
        for (int r = 0; r < n && !rc; ++r) rc = launch();
        if (!rc && hipEventRecord(b, s) != hipSuccess) rc = set_error(MOM6H_ESTATE, "event record failed");
        if (!rc && hipEventSynchronize(b) != hipSuccess) rc = set_error(MOM6H_ESTATE, "event wait failed");
        if (!rc && hipEventElapsedTime(&t, a, b) != hipSuccess) rc = set_error(MOM6H_ESTATE, "event timing failed");
        return t / (float)n;
    };
    // warm-up: about 6 ms; then timings of about 0.3 ms each
    const float first = std::max(time(0, 1), 1.0e-3f);
    const int warm = std::min(200, (int)(6.f / first)), per = first >= 0.3f ? 1 : std::min(16, (int)(0.3f / first) + 1);
    if (warm > 0) time(0, warm);
    float ms[N] = {}, best = 0.f;
    for (int round = 0; round < (reps > 1 ? reps : 1); ++round) {
        for (int c = 0; c < N; ++c) {
            const int q = round % 2 ? N - 1 - c : c;
            if (round > 0 && q != 0 && ms[q] > 1.05f * best) continue;   // out of the running
            const float t = time(q, per);
            if (round == 0 || t < ms[q]) ms[q] = t;
        }
        best = *std::min_element(ms, ms + N);
    }
    if (a) (void)hipEventDestroy(a);
    if (b) (void)hipEventDestroy(b);
    int pick = 0;
    for (int q = 1; q < N && !rc; ++q)
        if (ms[q] < 0.99f * ms[0] && (pick == 0 || ms[q] < ms[pick])) pick = q;
    const int rs = set(tile[pick], splits[pick]);
    rc = rc ? rc : rs;
    if (rc) return rc;
    auto name = [&](int q) { return q ? std::to_string(march_rows(tile[q], splits[q])) : std::string("auto"); };
    *report += "momentum march rows (ms, predictor + corrector):";
    for (int q = 0; q < N; ++q) {
        char buf[32];
        snprintf(buf, sizeof(buf), " %.4f;", ms[q]);
        *report += " " + name(q) + buf;
    }
    *report += " chosen " + name(pick);
    return MOM6H_OK;
}

// Del2u on u points I = is-1..ie, j = js..je and Del2v on v points i = is..ie,
// J = js-1..je (mom6_hor_visc_serial.F90:587-607), one thread per point with the
// march's expressions; runs only for a caller that reads the two fields
template <typename T>
__global__ void __launch_bounds__(256) k_del2(Del2Args<T> a)
{
    const Dims &d = a.d;
    const UMetT<T> g(a.g);
    const int i = d.isc - 1 + (int)blockIdx.x * 64 + (int)(threadIdx.x & 63);
    const int j = d.jsc - 1 + (int)blockIdx.y * 4 + (int)(threadIdx.x >> 6);
    const int k = 1 + (int)blockIdx.z;
    if (i > d.iec || j > d.jec) return;
    auto U = [&](int ii, int jj) -> T { return a.u[IX3(d, ii, jj, k)]; };
    auto V = [&](int ii, int jj) -> T { return a.v[IX3(d, ii, jj, k)]; };
    auto sh_xx = [&](int ii, int jj) -> T {   // h point (:503-510)
        const T dudx = g.DY_dxT * ((g.IdyCu * U(ii, jj)) - (g.IdyCu * U(ii - 1, jj)));
        const T dvdy = g.DX_dyT * ((g.IdxCv * V(ii, jj)) - (g.IdxCv * V(ii, jj - 1)));
        return dudx - dvdy;
    };
    auto sh_xy = [&](int I, int J) -> T {     // q point (:513-547)
        const T dvdx = g.DY_dxBu * ((V(I + 1, J) * g.IdyCv) - (V(I, J) * g.IdyCv));
        const T dudy = g.DX_dyBu * ((U(I, J + 1) * g.IdxCu) - (U(I, J) * g.IdxCu));
        const T m = (T)a.mask2dBu[IX2(d, I, J)];
        return (a.no_slip ? (T(2.0) - m) : m) * (dvdx + dudy);
    };
    const long long c = IX3(d, i, j, k);
    if (j >= d.jsc)
        a.del2u[c] = g.Idx2dyCu * ((g.dx2q * sh_xy(i, j)) - (g.dx2q * sh_xy(i, j - 1))) +
                     g.Idxdy2u * ((g.dy2h * sh_xx(i + 1, j)) - (g.dy2h * sh_xx(i, j)));
    if (i >= d.isc)
        a.del2v[c] = g.Idxdy2v * ((g.dy2q * sh_xy(i, j)) - (g.dy2q * sh_xy(i - 1, j))) -
                     g.Idx2dyCv * ((g.dx2h * sh_xx(i, j + 1)) - (g.dx2h * sh_xx(i, j)));
}

template <typename T>
int launch_del2(const Del2Args<T> &a, hipStream_t s)
{
    const Dims &d = a.d;
    k_del2<T><<<dim3((d.iec - d.isc + 2 + 63) / 64, (d.jec - d.jsc + 2 + 3) / 4, d.nk), 256, 0, s>>>(a);
    MOM6H_LAUNCH_CHECK();
    return MOM6H_OK;
}

template int launch_del2<double>(const Del2Args<double> &, hipStream_t);
template int launch_del2<float>(const Del2Args<float> &, hipStream_t);

// The masks as the stencil reads them, formed ahead of a step call when the fields
// were uploaded since, or when a caller holds the address of one and may have
// written it: 17 bytes per point of one plane, about 3 us at 720x720.
__global__ void __launch_bounds__(256) k_mask_bits(MaskJobs jobs)
{
    const MaskJob a = jobs.j[blockIdx.y];
    for (long long q = (long long)blockIdx.x * 256 + threadIdx.x; q < a.n; q += (long long)gridDim.x * 256)
        a.bits[q] = (unsigned char)((a.mask2dT[q] != 0.0 ? 1 : 0) | (a.mask2dBu[q] != 0.0 ? 2 : 0));
}

int launch_mask_bits(const MaskJobs &jobs, hipStream_t s)
{
    MOM6H_REQUIRE(jobs.n >= 1 && jobs.n <= kMaxMembers, "momentum masks: 1..%d grids", kMaxMembers);
    long long n = 1;
    for (int m = 0; m < jobs.n; ++m) n = std::max(n, jobs.j[m].n);
    k_mask_bits<<<dim3((unsigned)std::min(2048LL, (n + 255) / 256), jobs.n), 256, 0, s>>>(jobs);
    MOM6H_LAUNCH_CHECK();
    return MOM6H_OK;
}

template int launch_momentum<double>(const MomArgsT<double> &, hipStream_t);
template int launch_momentum<float>(const MomArgsT<float> &, hipStream_t);
template int plan_momentum_batch<double>(MomArgsT<double> *, int, int);
template int plan_momentum_batch<float>(MomArgsT<float> *, int, int);
template int launch_momentum_batch<double>(const MomArgsT<double> *, const MomArgsT<double> *, int, hipStream_t);
template int launch_momentum_batch<float>(const MomArgsT<float> *, const MomArgsT<float> *, int, hipStream_t);

}  // namespace mom6h
