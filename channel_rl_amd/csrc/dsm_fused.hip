// dsm_fused.hip -- dynamic Smagorinsky pass A in one kernel, FP64 (FP32:
// dsm_fp32.hip)
// (code/subgrid.f90:379-510): centre velocities, rate of strain |S| S_ij,
// filtered staggered velocities, the Leonard tensor L_ij, the model tensor
// M_ij and the per-row partial sums of L:M and M:M, plus |S| for pass B.
//
// Design: a block owns an x-y tile of CX x CY columns, one thread each, and
// marches in z.  A column takes what it needs of its x neighbours by cross-lane
// moves, of its y neighbours through LDS, and of the planes below from
// registers carried along the march, so every value crosses LDS once:
//   arrival of velocity plane q: the column's own U, V, W (registers) and the
//      rows above and below (LDS) give the y taps of the staggered test
//      filter and the plane's strain inputs (Plane below);
//   level 1 at plane q-1: centre velocities a and |S| S_ij, their products,
//      and the z taps of these 15 filter inputs (running sums in registers);
//      the z and x taps of the staggered filter;
//   LDS: the z-tapped filter inputs of plane q-2 and the filtered velocities
//      of plane q-1 go out, a barrier, the neighbouring rows come back;
//   output plane q-2: y and x taps of the filter inputs, hat(S) from the
//      filtered velocities (arriving plane by plane like the velocities),
//      L:M and M:M; the next velocity plane goes to LDS and the one after it
//      is fetched; a barrier.
// Columns include a halo of two in x (the outer one feeds the filtered
// velocities and strains of the inner one) and one in y: CX-4 x CY-2 outputs.
// The test filter is separable (y weights one-sided on rows 2 and nyg-1 as
// the reference).  Spacing divisions are multiplications by precomputed
// reciprocals.  The sums run in a different order than the reference, so the
// model agrees with it to rounding, not bit for bit.
// Global traffic: U,V,W read once per tile (plus halo), |S| written once.
// Measured (192x96x192): 106 us a launch against 142 before, when every operand of
// the strains and filters was read from LDS, from three velocity planes kept there:
// a wave's march of 40 planes issued 20,600 vector and 3,700 LDS instructions, now
// 17,700 and 2,100.  Bound by neither LDS (30% busy, no bank conflicts) nor the
// vector units (52%) but by the chain of a plane: two waves per SIMD, all the
// registers allow, take a plane in 2.3 us (106 us less 5 for the launch, over 44
// planes) where one alone takes 1.2 (12.7 less 3, over 8, at 32x32x32).
#include <algorithm>
#include <cmath>
#include "dsm.hpp"
#include "prof.hpp"

namespace chan {

// Planes per partial sum.  A block flushes its sums every DSM_SEG planes,
// counted from plane 2, and its chunk is a multiple of DSM_SEG: the partial
// sums, and with them <L:M>/<M:M>, do not depend on the chunk, so a grouped
// launch may take another one than a channel alone and still agree with it bit
// for bit.
constexpr int DSM_SEG = 4;

// Square root of a sum of squares x >= 0: the hardware reciprocal square
// root refined by the Newton-Raphson (Goldschmidt) steps of the library
// sequence, without its rescaling of tiny and huge arguments (a strain
// magnitude squared stays far inside the normal range; below 2^-960, where
// the hardware estimate would overflow, the result is 0, as for x = 0).
// Within an ulp of the correctly rounded root, in 13 instructions instead
// of the library's 17.
__device__ __forceinline__ double sqrt_sum_sq(double x)
{
    const double r = __builtin_amdgcn_rsq(x);
    double g = x * r, h = 0.5 * r;
    const double e = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, e, g);
    h = __builtin_fma(h, e, h);
    double d = __builtin_fma(-g, g, x);
    g = __builtin_fma(d, h, g);
    d = __builtin_fma(-g, g, x);
    g = __builtin_fma(d, h, g);
    return x > 0x1p-960 ? g : 0.0;
}


// sum over each 16 lanes of the wave, in its lane 15 (a fixed order); the
// whole wave must be active
__device__ __forceinline__ double row16_sum(double v)
{
    v += lane_shift<0x111>(v);  // row_shr:1, 2, 4, 8, zeros shifted in
    v += lane_shift<0x112>(v);
    v += lane_shift<0x114>(v);
    v += lane_shift<0x118>(v);
    return v;
}

// A segment of planes ends at k: a thread's sums of L:M and M:M over it, summed
// over each 16 columns of a row (CX columns per row, thread t in row t / CX,
// which is output row j0 - 1 + t / CX of rows 1..TYO) into b.part.  The whole
// wave must be active.
template <int CX, int TYO>
__device__ __forceinline__ void flush_segment(double lm, double mm, int t, int k, int j0, int tx, int gx, const Dims& d,
                                              const DsmBufs<double>& b)
{
    const double sl = row16_sum(lm), s2 = row16_sum(mm);
    asm("" : "+v"(t));  // the addresses are formed here, not held through the march
    const int r = t / CX, j = j0 - 1 + r;
    if (t % 16 == 15 && r >= 1 && r <= TYO && j <= d.nyg - 1) {
        const int blk = ((k - 2) / DSM_SEG * gx + tx) * (CX / 16) + t % CX / 16;
        double* o = b.part + (long)(j - 1) * 2 * b.nblk + blk;
        o[0] = sl;
        o[b.nblk] = s2;
    }
}

// What the strain at a plane k takes from the planes up to k, all of it this
// column's: with A(-1) the x neighbour below and A(j-1) the row below, the
// off-diagonal strains of code/subgrid.f90:1027-1070 (averages over the four
// surrounding edges of (dA/db + dB/da)/2) group into
//   S12 = 1/8 (eU + eU(-1) + rx0 (vs - vs(-1)) + rx1 (vs(+1) - vs)),
//   S13 = 1/8 (t + t(-1) + rx0 (ws - ws(-1)) + rx1 (ws(+1) - ws)),
//         t = rz0 (U - U(k-1)) + rz1 (U(k+1) - U),  ws = W(k-1) + W,
//   S23 = 1/8 (rz0 (vs - vs(k-1)) + rz1 (vs(k+1) - vs) + eW(k-1) + eW),
// seven cross-lane moves and no neighbour row beyond those in eU, vs and eW.
// The factor 1/8 is in the spacings r0, r1 (Met3), which enter nowhere else.
struct Plane {
    double u;    // U
    double eU;   // ry0 (U - U(j-1)) + ry1 (U(j+1) - U)
    double vs;   // V(j-1) + V
    double vd;   // V - V(j-1)
    double w;    // W
    double wb;   // W(k-1)
    double eW;   // ry0 (W - W(j-1)) + ry1 (W(j+1) - W)
    double t13;  // rz0 (U - U(k-1))
    double t23;  // rz0 (vs - vs(k-1)) + eW(k-1) + eW
};

// reciprocal spacings of a column: r = 1/(x(i)-x(i-1)), r0 = 1/8 / (xg(i)-xg(i-1)),
// r1 = 1/8 / (xg(i+1)-xg(i)), the same in y; per plane in z
struct Met3 { double r, r0, r1; };

// plane k from (U, V, W) at rows j, j-1, j+1 and the plane below it; rz0 =
// 1/8 / (zg(k)-zg(k-1))
__device__ __forceinline__ Plane arrive(const double (&o)[3], const double (&m)[3], const double (&n)[3], const Plane& below,
                                           const Met3& y, double rz0)
{
    Plane p;
    p.u = o[0];
    p.eU = y.r0 * (o[0] - m[0]) + y.r1 * (n[0] - o[0]);
    p.vs = m[1] + o[1];
    p.vd = o[1] - m[1];
    p.w = o[2];
    p.wb = below.w;
    p.eW = y.r0 * (o[2] - m[2]) + y.r1 * (n[2] - o[2]);
    p.t13 = rz0 * (o[0] - below.u);
    p.t23 = rz0 * (p.vs - below.vs) + (below.eW + p.eW);
    return p;
}

// s: S11, S22, S33, S12, S13, S23 at plane p, q the plane above; uL: U(-1)
__device__ __forceinline__ void strain(const Plane& p, const Plane& q, const Met3& x, double ry, double rz, double rz1,
                                       double (&s)[6], double& uL)
{
    uL = lane_shift<DPP_WAVE_SHR1>(p.u);
    const double ws = p.wb + p.w;
    s[0] = (p.u - uL) * x.r;
    s[1] = p.vd * ry;
    s[2] = (p.w - p.wb) * rz;
    const double vl = lane_shift<DPP_WAVE_SHR1>(p.vs), vr = lane_shift<DPP_WAVE_SHL1>(p.vs);
    const double wl = lane_shift<DPP_WAVE_SHR1>(ws), wr = lane_shift<DPP_WAVE_SHL1>(ws);
    const double t = p.t13 + rz1 * (q.u - p.u);
    s[3] = (p.eU + lane_shift<DPP_WAVE_SHR1>(p.eU)) + x.r0 * (p.vs - vl) + x.r1 * (vr - p.vs);
    s[4] = (t + lane_shift<DPP_WAVE_SHR1>(t)) + x.r0 * (ws - wl) + x.r1 * (wr - ws);
    s[5] = p.t23 + rz1 * (q.vs - p.vs);
}
// |S| = sqrt(2 S_ij S_ij)
__device__ __forceinline__ double magnitude(const double (&s)[6])
{
    const double dg = s[0] * s[0] + s[1] * s[1] + s[2] * s[2];
    const double od = s[3] * s[3] + s[4] * s[4] + s[5] * s[5];
    return sqrt_sum_sq(2.0 * (dg + 2.0 * od));
}

// Planes in LDS are 16-byte vectors: a wave's ds_read_b128 takes half the time
// of the paired ds_read2st64_b64 that planes of single values become (16 values
// a lane, four waves: 58 against 108 ns measured).
typedef double V2 __attribute__((ext_vector_type(2)));
// a plane P of n positions of staggered velocities: (U, W) pairs, then V
__device__ __forceinline__ int vel_at(int n, int q, int f) { return f == 1 ? 2 * n + q : 2 * q + (f >> 1); }
__device__ __forceinline__ void vel_get(const double* P, int n, int q, double (&u)[3])
{
    const V2 a = ((const V2*)P)[q];
    u[0] = a.x;
    u[1] = P[2 * n + q];
    u[2] = a.y;
}
__device__ __forceinline__ void vel_put(double* P, int n, int q, double u, double v, double w)
{
    ((V2*)P)[q] = V2{u, w};
    P[2 * n + q] = v;
}

// DT: also compute_dt's maxima over the block's output cells, into b.dtpart
template <int CX, int CY, bool G, bool DT>
__global__ void __launch_bounds__(CX* CY) __attribute__((amdgpu_waves_per_eu(2)))
    k_dsm_fused(DsmArgs<double> one, const DsmArgs<double>* tab, Dims d, int kchunk)
{
    // The model's sums are reordered against the reference anyway (separable
    // filter, per-row partials); contracting a*b+c into FMAs here saves a
    // third of the FP64 instructions and changes results only by rounding.
#pragma clang fp contract(fast)
    constexpr int NT = CX * CY, TXO = CX - 4, TYO = CY - 2, NL = CX * (CY + 2);
    static_assert(64 % CX == 0 && CX % 16 == 0 && NT % 64 == 0, "rows of columns must tile the waves");
    static_assert(6 * CX <= NT, "one thread per value of the two outer rows");
    // LDS planes, in one array so that a row offset from the first or last row
    // of one stays inside it (such values are not used)
    __shared__ __attribute__((aligned(16))) double sm_all[3 * (NL + NT) + 16 * NT];
    double* const l0 = sm_all;        // velocities: rows -1..CY of the tile's columns
    double* const lf = l0 + 3 * NL;   // filtered velocities (times 216)
    V2* const Z = (V2*)(lf + 3 * NT) + threadIdx.x;  // z-tapped filter inputs in pairs: a(3), a_a a_b (6), |S|S_ij (6)
    __shared__ double mz[3][DSM_KMAX + 5];      // Met3 in z of plane p = kb-3+q
    __shared__ double mxt[3][CX];               // Met3 in x at the true index of the outputs
    __shared__ double mzd[DT ? DSM_KMAX + 5 : 1];  // zg(p+1) - zg(p), for compute_dt

    const int tid = threadIdx.x;
    const int cx = tid % CX, cy = tid / CX;
    const GBlk gb = gblk_xcd((d.nzg - 2 + kchunk - 1) / kchunk);
    const DsmArgs<double> arg = member_args<G>(one, tab, gb.m);
    const DsmBufs<double> b = arg.b;
    const TileId tile{gb.x, gb.y, gb.z};
    const int i0 = tile.x * TXO + 2, j0 = tile.y * TYO + 2;
    const int kb = tile.z * kchunk + 2;
    const int ke = min(kb + kchunk - 1, d.nzg - 1);
    const int ci = i0 - 2 + cx, cj = j0 - 1 + cy;  // column position (x unwrapped)
    const int nxp = d.nxp, nzp = d.nzp;
    // periodic wrap onto the unique points 2..nxp+1.  The columns an output
    // reads are within one period of that range; those beyond (a tile wider
    // than the rest of the row) read the last one and are not used.
    auto wx = [&](int q) { return q < 2 ? q + nxp : (q > nxp + 1 ? min(q - nxp, nxp + 1) : q); };
    auto wz = [&](int q) { return q < 2 ? q + nzp : (q > nzp + 1 ? q - nzp : q); };
    const double h = 0.5;
    // z reciprocal spacings of the block's planes, in LDS: a global load per
    // plane would wait behind the velocity prefetch (memory counters drain in
    // issue order).  Level 1 uses the canonical images, the outputs the true
    // index (code/subgrid.f90:456), which on output planes are the same.
    const double e8 = 0.125;
    for (int q = tid; q < ke - kb + 6; q += NT) {
        const int pc = wz(kb - 3 + q);
        mz[0][q] = b.rdz[pc];
        mz[1][q] = e8 * b.rdzg[pc];
        mz[2][q] = e8 * b.rdzg[pc + 1];
        if (DT) mzd[q] = b.zg[pc + 1] - b.zg[pc];
    }
    if (tid < CX) {
        const int it = min(max(ci, 2), d.nxg - 1);
        mxt[0][tid] = b.rdx[it];
        mxt[1][tid] = e8 * b.rdxg[it];
        mxt[2][tid] = e8 * b.rdxg[it + 1];
    }
    const int ic = wx(ci), jt = min(max(cj, 2), d.nyg - 1);
    const Met3 mxc{b.rdx[ic], e8 * b.rdxg[ic], e8 * b.rdxg[ic + 1]};
    const Met3 my{b.rdy[jt], e8 * b.rdyg[jt], e8 * b.rdyg[jt + 1]};

    // Global loads: every thread its own column of U, V, W, and 6 CX threads
    // one value each of the rows below and above the tile's columns (U, V, W
    // of row -1, then of row CY).  The staggered filter is one-sided at the
    // first and last row of each field (weights (0, 4, 2) and (2, 4, 0),
    // code/subgrid.f90:140-190): the row beyond either is loaded as its mirror
    // image, so that both taps of those rows read their inner neighbour.  The
    // strains of those rows either do not use it (V's last row) or are not
    // used (the wall ghost rows); rows further out are clamped and not used.
    auto row = [&](int j, int n) { return j == 0 ? 2 : (j == n + 1 ? n - 1 : min(max(j, 1), n)); };
    // byte offsets within a plane (below 2^32: the box's 2^31 values are in at
    // least seven planes), added to the plane's uniform base address
    auto bytes = [&](int i, int j) { return (unsigned)(at(d, i, j, 1) * sizeof(double)); };
    auto ld = [&](const double* base, unsigned o) { return *(const double*)((const char*)base + o); };
    unsigned own = bytes(ic, row(cj, d.nyg)), ownv = bytes(ic, row(cj, d.ny));
    // the outer value's field and row; one field per wave where a wave holds
    // two rows
    const int xf = CX == 32 ? __builtin_amdgcn_readfirstlane(tid / 64) : tid / (2 * CX), xr = (tid / CX) % 2;
    const bool has_x = tid < 6 * CX;
    unsigned ext = bytes(ic, row(xr == 0 ? j0 - 2 : j0 - 1 + CY, xf == 1 ? d.ny : d.nyg));
    const double* const xsrc = xf == 1 ? arg.V : (xf == 2 ? arg.W : arg.U);
    double pu, pv, pw, px;  // the plane in flight
    auto gload = [&](int p) {
        // (the opaque offsets keep the addresses out of register pairs per
        // lane: a scalar base per plane plus 32 bits)
        asm("" : "+v"(own), "+v"(ownv), "+v"(ext));
        const long po = (long)(wz(p) - 1) * d.sxy;
        pu = ld(arg.U + po, own);
        pv = ld(arg.V + po, ownv);
        pw = ld(arg.W + po, own);
        px = ld(xsrc + po, ext);
    };
    const int qo = cx + CX * (cy + 1);  // own position in l0
    auto sstore = [&]() {
        vel_put(l0, NL, qo, pu, pv, pw);
        if (has_x) l0[vel_at(NL, cx + (xr == 0 ? 0 : CX * (CY + 1)), xf)] = px;
    };
    // rows for the y taps of the filter inputs, one-sided at rows 2 and nyg-1;
    // the halo rows 0 and CY-1 take taps as well and do not use them
    const int qm = cj == 2 ? CX : -CX, qp = cj == d.nyg - 1 ? -CX : (cy == CY - 1 ? 0 : CX);

    const bool out_col = cx >= 2 && cx < 2 + TXO && cy >= 1 && cy <= TYO && ci <= d.nxg - 1 && cj <= d.nyg - 1;
    const bool st_col = out_col && ci <= nxp + 1;  // a unique cell: |S| goes there and to its images
    // compute_dt over this column's output cells (DT): the
    // smallest |U| and |V| (x and y spacings are the column's own, and a
    // correctly rounded quotient falls as its divisor grows, so the largest
    // dx/|U| is dx over the smallest |U|, exactly), and the largest dz/|W|
    // plane by plane (the z spacings differ in their last bits)
    // (in LDS, each thread its own slots: the march has no registers left)
    __shared__ double dt_mu[DT ? NT : 1], dt_mv[DT ? NT : 1];
    __shared__ double dt_lw[DT ? NT : 1];
    if constexpr (DT) {
        dt_mu[tid] = dt_mv[tid] = INFINITY;
        dt_lw[tid] = 0.0;
    }
    constexpr int pa[6] = {0, 1, 2, 0, 0, 1}, pb[6] = {0, 1, 2, 1, 2, 2};

    double acc_lm = 0.0, acc_mm = 0.0;
    Plane vel{}, fil{};     // the last plane of the velocities and of the filtered ones
    double fA[3] = {}, fB[3] = {};  // staggered filter: y taps of the last plane, running z sum
    double fC[3] = {};

    // One arriving velocity plane q (q - 2 the output plane).  The z taps run as
    // sums over three arrays whose roles rotate (no register copies): za holds
    // Q(q-3) + 4 Q(q-2) and becomes the tapped plane q-2, zb Q(q-2) and becomes
    // Q(q-2) + 4 Q(q-1), zc receives Q(q-1) (the planes before the chunk run
    // through the same code without a branch: what they leave in the sums is
    // rotated out before it is used); the same for the staggered filter
    // with the y taps Y(q): ya = Y(q-2) + 4 Y(q-1), yb = Y(q-1).
    auto step = [&](int q, double (&za)[15], double (&zb)[15], double (&zc)[15], double (&ya)[3], double (&yb)[3], double (&yc)[3]) {
        const int p = q - 1, k = q - 2;
        {
            double o[3], m[3], n[3];  // U, V, W: own row, the rows below and above
            vel_get(l0, NL, qo, o);
            vel_get(l0, NL, qo - CX, m);
            vel_get(l0, NL, qo + CX, n);
            for (int f = 0; f < 3; f++) yc[f] = (m[f] + n[f]) + 4.0 * o[f];
            if constexpr (DT) {
                if (out_col && q >= kb && q <= ke) {
                    dt_mu[tid] = fmin(dt_mu[tid], fabs(o[0]));
                    dt_mv[tid] = fmin(dt_mv[tid], fabs(o[1]));
                    dt_lw[tid] = fmax(dt_lw[tid], mzd[q - kb + 3] / fabs(o[2]));
                }
            }
            const Plane nxt = arrive(o, m, n, vel, my, mz[1][q - kb + 3]);
            // (keeps the scheduler from interleaving the stages, which costs
            // more registers than two waves per SIMD have)
            __builtin_amdgcn_sched_barrier(0);
            {
                // level 1 of this column at plane p: the filter inputs a (3),
                // a_a a_b (6), |S| S_ij (6).  Rows outside 2..nyg-1 compute on
                // the mirrored or clamped rows loaded there and finite metric
                // factors, and are not used: the y taps of rows 2 and nyg-1 read
                // their inner neighbour for both (qm, qp).
                double s[6], uL;
                strain(vel, nxt, mxc, my.r, mz[0][p - kb + 3], mz[2][p - kb + 3], s, uL);
                const double sm = magnitude(s);
                if (p >= kb && p <= min(ke, nzp + 1)) {
                    int t = tid;
                    asm("" : "+v"(own), "+v"(t));
                    if (st_col) store_smag(b.smag, d, p, own, i0 - 2 + t % CX, sm);
                }
                // code/subgrid.f90:394-396 centre velocities
                zc[0] = h * (uL + vel.u);
                zc[1] = h * vel.vs;
                zc[2] = h * (vel.wb + vel.w);
#pragma unroll
                for (int c = 0; c < 6; c++) {
                    zc[3 + c] = zc[pa[c]] * zc[pb[c]];
                    zc[9 + c] = sm * s[c];
                }
#pragma unroll
                for (int g = 0; g < 8; g++) {
                    V2 t;
#pragma unroll
                    for (int e = 0; e < 2; e++) {
                        const int c = 2 * g + e;
                        t[e] = 0.0;
                        if (c < 15) {
                            // each product once, not again inside the sums' FMAs
                            asm("" : "+v"(zc[c]));
                            t[e] = za[c] + zc[c];
                            zb[c] = zb[c] + 4.0 * zc[c];
                        }
                    }
                    Z[g * NT] = t;
                }
                // filtered velocities of plane p: z taps done, x taps here
                double y[3];
#pragma unroll
                for (int f = 0; f < 3; f++) {
                    const double t = ya[f] + yc[f];
                    y[f] = (lane_shift<DPP_WAVE_SHR1>(t) + lane_shift<DPP_WAVE_SHL1>(t)) + 4.0 * t;
                }
                vel_put(lf, NT, tid, y[0], y[1], y[2]);
            }
            vel = nxt;
        }
#pragma unroll
        for (int f = 0; f < 3; f++) yb[f] = yb[f] + 4.0 * yc[f];
        __syncthreads();
        if (q <= ke + 1) {
            sstore();
            if (q <= ke) gload(q + 2);
        }
        {
            // the filtered plane p arrives
            double o[3], m[3], n[3];
            vel_get(lf, NT, tid, o);
            vel_get(lf, NT, tid - CX, m);
            vel_get(lf, NT, tid + CX, n);
            const Plane nxt = arrive(o, m, n, fil, my, mz[1][p - kb + 3]);
            if (k >= kb) {
                // hat(S), 216 times, at the true index (code/subgrid.f90:456)
                const Met3 x{mxt[0][cx], mxt[1][cx], mxt[2][cx]};
                double sh[6], uL;
                strain(fil, nxt, x, my.r, mz[0][k - kb + 3], mz[2][k - kb + 3], sh, uL);
                __builtin_amdgcn_sched_barrier(0);
                // x-y taps of the 15 filter inputs, every lane (cross-lane moves)
                double tp[15];
#pragma unroll
                for (int g = 0; g < 8; g++) {
                    // (the own value from LDS again: its registers are needed)
                    const V2 o = Z[g * NT], m = Z[g * NT + qm], n = Z[g * NT + qp];
#pragma unroll
                    for (int e = 0; e < 2; e++) {
                        const int c = 2 * g + e;
                        if (c < 15) {
                            const double y = (m[e] + n[e]) + 4.0 * o[e];
                            tp[c] = (lane_shift<DPP_WAVE_SHR1>(y) + lane_shift<DPP_WAVE_SHL1>(y)) + 4.0 * y;
                        }
                    }
                }
                // tp holds 216 times the filtered inputs and sh 216 times
                // hat(S): with r = 1/216, L = r (T_ab - r T_a T_b) and
                // M = 4 |hat S| hat S_ab - r T(|S| S_ab) = r (4 r |sh| sh_ab - T(|S| S_ab)),
                // the outer factors taken once on the sums
                const double r = 1.0 / 216.0;
                const double shm4 = (4.0 * r) * magnitude(sh);
                const double sa[3] = {r * tp[0], r * tp[1], r * tp[2]};
                double lm = 0.0, mm = 0.0;
#pragma unroll
                for (int e = 0; e < 6; e++) {
                    const double L = tp[3 + e] - sa[pa[e]] * tp[pb[e]];
                    const double M = shm4 * sh[e] - tp[9 + e];
                    const double wgt = e < 3 ? 1.0 : 2.0;
                    lm = lm + wgt * (L * M);
                    mm = mm + wgt * (M * M);
                }
                acc_lm += out_col ? (r * r * lm) : 0.0;
                acc_mm += out_col ? (r * r * mm) : 0.0;
                if ((k - 1) % DSM_SEG == 0 || k == ke) {
                    flush_segment<CX, TYO>(acc_lm, acc_mm, tid, k, j0, tile.x, gb.gx, d, b);
                    acc_lm = 0.0;
                    acc_mm = 0.0;
                }
            }
            fil = nxt;
        }
        __syncthreads();
    };

    double zA[15] = {}, zB[15] = {}, zC[15] = {};
    gload(kb - 2);
    sstore();
    gload(kb - 1);
    __syncthreads();
    // planes kb-2..ke+2, unrolled by three so that the sums' arrays rotate
    // without copies
    for (int q = kb - 2;;) {
        step(q, zA, zB, zC, fA, fB, fC);
        if (++q > ke + 2) break;
        step(q, zB, zC, zA, fB, fC, fA);
        if (++q > ke + 2) break;
        step(q, zC, zA, zB, fC, fA, fB);
        if (++q > ke + 2) break;
    }
    if constexpr (DT) {
        double m3[3] = {0.0, 0.0, dt_lw[tid]};
        if (out_col) {
            m3[0] = (b.xg[ci + 1] - b.xg[ci]) / dt_mu[tid];
            m3[1] = (b.yg[cj + 1] - b.yg[cj]) / dt_mv[tid];
        }
        __shared__ double wmax[NT / 64][3];
        dt_block_maxima<NT>(m3, wmax, tid, gb, b);
    }
}

// A tile shape: columns and outputs in x and y, resident blocks per CU.
struct DsmTile { int cx, cy, tx, ty, per_cu; };

// Estimated time of one launch in us: nb blocks of a tile marching kc planes.
// A plane takes sqrt(l^2 + (t w)^2) us with w waves on a SIMD (l: one wave's
// chain of dependent steps, t: what each further wave costs), a block its planes
// plus `pre` (the pre-roll and the first loads), and blocks beyond the resident
// ones wait for a place.
double dsm_cost(const DsmTile& q, long nb, int kc, int ncu, double l, double t, double pre)
{
    const double deep = (double)((nb + ncu - 1) / ncu);  // blocks per CU
    const double c = std::min(deep, (double)q.per_cu);
    const double w = c * q.cx * q.cy / 256.0;
    return (kc + pre) * std::sqrt(l * l + t * w * t * w) * deep / c;
}

// The tile (of the three, or the given one) and chunk with the least estimate
// for nmem channels in one launch
DsmPlan dsm_pick(const DsmTile (&tiles)[3], double l, double t, double pre, const Dims& d, int device, int shape,
                        int nmem)
{
    int ncu = 0;
    if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || ncu < 1) ncu = 1;
    const int nk = d.nzg - 2;
    DsmPlan best{};
    double bc = -1.0;
    for (int q = 1; q <= 3; q++) {
        if (shape > 0 && q != shape) continue;
        const DsmTile& ti = tiles[q - 1];
        const int gx = cdiv(d.nxg - 2, ti.tx);
        const long xy = (long)gx * cdiv(d.nyg - 2, ti.ty);
        for (int kc = DSM_SEG; kc <= DSM_KMAX; kc += DSM_SEG) {
            const double c = dsm_cost(ti, xy * cdiv(nk, kc) * nmem, std::min(kc, nk), ncu, l, t, pre);
            if (bc >= 0.0 && c >= bc) continue;
            bc = c;
            best = DsmPlan{q, kc, gx * (ti.cx / 16) * cdiv(nk, DSM_SEG), (int)(xy * cdiv(nk, kc))};
        }
    }
    return best;
}

// Tile shapes: shape 0 takes whichever of 1..3 the estimate puts first for the
// grid.  l, t and the pre-roll are fitted to a sweep over tiles and chunks on
// grids from 32x32x32 to 384x192x384, which they reproduce within about 10%;
// the best pairs of the sweep were
//   32x32x32     tile 3 chunk 4   12.7 us (tile 1: 18.0)
//   64x48x64     tile 3 chunk 4   18.3 us (tile 1: 19.1)
//   128x40x64    tile 1 chunk 4   19.8 us (tile 3: 26.8)
//   192x96x192   tile 1 chunk 40 105.9 us (tile 2: 123, tile 3: 144)
//   384x192x384  tile 1 chunk 40 803 us   (tile 2: 822, tile 3: 932)
template <int CX, int CY>
DsmTile dsm_tile()
{
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_dsm_fused<CX, CY, false, false>, CX * CY, 0) != hipSuccess ||
        n < 1)
        n = 1;
    return DsmTile{CX, CY, CX - 4, CY - 2, n};
}

template <>
DsmPlan dsm_plan<double>(const Dims& d, int device, int shape, int nmem)
{
    // (the same on every gfx950: asked once)
    static const DsmTile tiles[3] = {dsm_tile<32, 16>(), dsm_tile<32, 8>(), dsm_tile<16, 8>()};
    return dsm_pick(tiles, 1.55, 0.87, 3.2, d, device, shape, nmem);
}

int dsm_shape_count() { return 4; }

template <>
void run_dsm_fused<double>(const DsmArgs<double>& one, const DsmArgs<double>* tab, int nmem, const Dims& d, int kchunk,
                           int tile, hipStream_t s)
{
    dsm_check(kchunk, tile, 1);
    PROF_BEGIN("k_dsm_fused", s);
#define DSM_GO(CX, CY)                                                                                             \
    do {                                                                                                           \
        const dim3 grd(cdiv(d.nxg - 2, CX - 4), cdiv(d.nyg - 2, CY - 2), (unsigned)cdiv(d.nzg - 2, kchunk) * nmem); \
        if (tab) k_dsm_fused<CX, CY, true, false><<<grd, CX * CY, 0, s>>>(one, tab, d, kchunk);                     \
        else if (one.b.dtpart) k_dsm_fused<CX, CY, false, true><<<grd, CX * CY, 0, s>>>(one, tab, d, kchunk);       \
        else k_dsm_fused<CX, CY, false, false><<<grd, CX * CY, 0, s>>>(one, tab, d, kchunk);                        \
    } while (0)
    if (tile == 1) DSM_GO(32, 16);
    else if (tile == 2) DSM_GO(32, 8);
    else DSM_GO(16, 8);
#undef DSM_GO
    PROF_END(s);
}

}  // namespace chan
