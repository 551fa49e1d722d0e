// tb_helm.hip -- Helmholtz operators of the momentum and concentration
// predictors and their BiCGStab solve, all matrix-free on the device.
//
// Rows follow Velocity_u/v/w_form_LHS_matrix (Velocity.c:449-1471) and
// Conc_form_LHS_matrix (Conc.c:390-730) term by term, with the diagonal
// update of Velocity_modify_diagonal / Conc_modify_diagonal
// (Velocity.c:374-443, Conc.c:293-354) added to every non-IMMERSED row.
// Each row is summed in ascending column order, as PETSc's AIJ MatMult
// does, so one application is bit-identical to the assembled matrix's.
//
// The operator kernel walks k inside each column tile: the x and y parts of
// every coefficient are formed once per column, the z parts once per plane
// (uniform across the block), and the k-1 / k / k+1 values stay in
// registers.  The neighbour-status tests of the reference reduce to index
// tests, because BOUNDARY nodes are exactly the box planes.
#include <cmath>
#include <utility>

#include "tb_common.h"

struct HelmOp {
    Dims d;
    GridDev g;
    int q;
    const uint8_t *st;
    double Cx, Cy, Cz, ap_solid, mod;
    int wall[6];
    int particle;
    double robin_b_scale;   // 2/(Pe*dXi)
    double vs_abs;
    // open x faces drop their wall rule: c at x = 0 with inflow, v, w and c
    // at x = Lx with outflow (Velocity.c:989, 1336; Conc.c:582-607)
    int open_w, open_e;
};

// What the Gauss-Seidel kernels need of one quantity's solve.  u, v, w and
// the concentration fields are solved side by side, one grid row (blockIdx.y)
// each: their systems are independent, and one quantity's launches leave much
// of the chip idle.
struct GsView {
    HelmOp H;
    const double *b, *x0;          // right-hand side; the field the solve started from
    const double *from;            // iterate read and iterate written by a pair
    double *to;
    const float *inc;              // increment added to `from` (none: null)
    float *dn;                     // increment to - x0, written by the residual check
    const long *row, *col;         // IMMERSED rows (ib_row, ...)
    const int *cnt;
    const double *val;
    int nib;
};

constexpr int HELM_SET = 3 + TB_NCONC_MAX;

template <int N>
struct GsSet {   // a kernel argument: at most 4 KB
    GsView v[N];
    __device__ const GsView &mine() const { return v[N == 1 ? 0 : blockIdx.y]; }
};

// k_helm_check's argument list is the longest; the runtime's own arguments
// follow in the same segment
static_assert(sizeof(GsSet<HELM_SET>) + sizeof(double *) + sizeof(long) + sizeof(KTiles) <= 4096 - 256,
              "kernel arguments");

// wall rule applied to ap when a neighbour is absent:
// 0 nothing (normal component on the wall), 1 no-slip (ap -= a),
// 2 free-slip / Neumann (ap += a)
__device__ inline double wallmod(double ap, double a, int rule) {
    if (rule == 1) return ap - a;
    if (rule == 2) return ap + a;
    return ap;
}

// MODE 0: y = A x ; MODE 1: also partial w.y ; MODE 2: also partials x.y, y.y
// MODE 3: residual only: partials |w - A x|^2 and |w|^2 with w = b, nothing
// stored (IMMERSED rows must hold (A x) from k_ib_apply in y), and the
// increment dn = x - x0 over the box (the Gauss-Seidel solve's change to the
// field it started from).
// IMMERSED rows are produced by k_ib_apply, which runs first; here their y is
// only read for the dot products.
template <int MODE>
__device__ __forceinline__ void helm_rows(const HelmOp &H, const double *__restrict__ x, double *__restrict__ y,
                                          const double *__restrict__ w, double *part, const KTiles &t,
                                          const double *__restrict__ x0, float *__restrict__ dn) {
    __shared__ double sh[32];
    double acc[2] = {0.0, 0.0};
    int i, j, k0, k1;
    bool act;
    ktile_column(t, i, j, k0, k1, act);
    if (act) {
        const Dims &d = H.d;
        const GridDev &g = H.g;
        const int NX = d.NX, NY = d.NY, NZ = d.NZ;
        const int q = H.q;
        const double Cx = H.Cx, Cy = H.Cy, Cz = H.Cz;
        const int im1 = i > 0 ? i - 1 : 0, ip1 = i + 1 < NX ? i + 1 : NX - 1;
        const int jm1 = j > 0 ? j - 1 : 0, jp1 = j + 1 < NY ? j + 1 : NY - 1;
        double mpx, mex, mwx, mpy, mny, msy;
        if (q == TB_Q_U) {
            mpx = g.mxu[i]; mex = g.mxc[i]; mwx = g.mxc[im1]; mpy = g.myc[j]; mny = g.myv[jp1]; msy = g.myv[j];
        } else if (q == TB_Q_V) {
            mpx = g.mxc[i]; mex = g.mxu[ip1]; mwx = g.mxu[i]; mpy = g.myv[j]; mny = g.myc[j]; msy = g.myc[jm1];
        } else {
            mpx = g.mxc[i]; mex = g.mxu[ip1]; mwx = g.mxu[i]; mpy = g.myc[j]; mny = g.myv[jp1]; msy = g.myv[j];
        }
        // ((-Cx mpx (mex+mwx)) - Cy mpy (mny+msy)) - Cz mpz (mbz+mfz), left to right
        const double axy = -Cx * mpx * (mex + mwx) - Cy * mpy * (mny + msy);
        const double aw = Cx * mpx * mwx, ae = Cx * mpx * mex;
        const double an = Cy * mpy * mny, as = Cy * mpy * msy;
        // per-column presence and wall rules of the x and y neighbours
        bool hs, hw, he, hn;
        int rs, rw, re, rn;
        const int *W = H.wall;
        if (q == TB_Q_U) {
            hs = j != 0;       rs = W[2] ? 1 : 2;
            hw = i - 1 >= 1;   rw = 0;
            he = i + 1 <= NX - 2; re = 0;
            hn = j != NY - 2;  rn = W[3] ? 1 : 2;
        } else if (q == TB_Q_V) {
            hs = j - 1 >= 1;   rs = 0;
            hw = i != 0;       rw = W[0] ? 1 : 2;
            he = i < NX - 2;   re = (i == NX - 2) ? (H.open_e ? 0 : (W[1] ? 1 : 2)) : 0;
            hn = j + 1 <= NY - 2; rn = 0;
        } else if (q == TB_Q_W) {
            hs = j != 0;       rs = W[2] ? 1 : 2;
            hw = i != 0;       rw = W[0] ? 1 : 2;
            he = i < NX - 2;   re = (i == NX - 2) ? (H.open_e ? 0 : (W[1] ? 1 : 2)) : 0;
            hn = j != NY - 2;  rn = W[3] ? 1 : 2;
        } else {
            hs = j > 0;        rs = 2;
            hw = i > 0;        rw = H.open_w ? 0 : 2;
            he = i < NX - 2;   re = H.open_e ? 0 : 2;
            hn = j < NY - 2;   rn = 2;
        }
        double cn = an;   // north wall term (Robin for settling particles, Conc.c:625-635)
        if (q == TB_Q_C && H.particle) {
            double b = H.robin_b_scale * mny;
            cn = an * (b - H.vs_abs) / (b + H.vs_abs);
        }
        const int rb = (q == TB_Q_W) ? 0 : (q == TB_Q_C ? 2 : (W[4] ? 1 : 2));
        const int rf = (q == TB_Q_W) ? 0 : (q == TB_Q_C ? 2 : (W[5] ? 1 : 2));
        const bool row_buffer = (q != TB_Q_C);   // BUFFER_SOLID rows carry the stencil for u, v, w
        const double diag_other = H.ap_solid + H.mod;

        // neighbour offsets clamped to the point itself at the box faces, so
        // every load is issued unconditionally and the loads overlap
        const long os = (j > 0) ? d.px : 0, on = (j + 1 < NY) ? d.px : 0;
        const long ow = (i > 0) ? 1 : 0, oe = (i + 1 < NX) ? 1 : 0;
        long id = gidx(d, i, j, k0);
        double xm = x[id - ((k0 > 0) ? d.plane : 0)];
        double xc = x[id];
        for (int k = k0; k < k1; k++) {
            double xp = x[id + ((k + 1 < NZ) ? d.plane : 0)];
            const double xs = x[id - os], xw = x[id - ow], xe = x[id + oe], xn = x[id + on];
            const double wv = (MODE == 1 || MODE == 3) ? __builtin_nontemporal_load(&w[id]) : 0.0;
            const double x0v = (MODE == 3) ? __builtin_nontemporal_load(&x0[id]) : 0.0;
            const int s = H.st[id];
            // the fluid row is formed for every node and selected afterwards:
            // no status-dependent branch sits between the loads and the math
            const int km1 = k > 0 ? k - 1 : 0, kp1 = k + 1 < NZ ? k + 1 : NZ - 1;
            double mpz, mbz, mfz;
            if (q == TB_Q_W) { mpz = g.mzw[k]; mbz = g.mzc[km1]; mfz = g.mzc[k]; }
            else { mpz = g.mzc[k]; mbz = g.mzw[k]; mfz = g.mzw[kp1]; }
            double ap = axy - Cz * mpz * (mbz + mfz);
            const double ab = Cz * mpz * mbz, af = Cz * mpz * mfz;
            bool hb, hf;
            if (q == TB_Q_W) { hb = k - 1 >= 1; hf = k + 1 <= NZ - 2; }
            else if (q == TB_Q_C) { hb = k > 0; hf = k < NZ - 2; }
            else { hb = k != 0; hf = k != NZ - 2; }
            // wall terms in the reference's order: back, south, west, east, north, front
            if (!hb) ap = wallmod(ap, ab, rb);
            if (!hs) ap = wallmod(ap, as, rs);
            if (!hw) ap = wallmod(ap, aw, rw);
            if (!he) ap = wallmod(ap, ae, re);
            if (!hn) ap = (q == TB_Q_C) ? ap + cn : wallmod(ap, an, rn);
            if (!hf) ap = wallmod(ap, af, rf);
            double r = 0.0;
            r = hb ? r + ab * xm : r;
            r = hs ? r + as * xs : r;
            r = hw ? r + aw * xw : r;
            r += (ap + H.mod) * xc;
            r = he ? r + ae * xe : r;
            r = hn ? r + an * xn : r;
            r = hf ? r + af * xp : r;
            const bool fluid = (s == TB_FLUID) || (row_buffer && s == TB_BUFFER_SOLID);
            double yv = fluid ? r : diag_other * xc;
            if (s == TB_IMMERSED) {
                yv = (MODE > 0) ? y[id] : 0.0;   // row written by k_ib_apply
            } else if (MODE < 3) {
                st_stream(&y[id], yv);
            }
            if (MODE == 3) st_stream(&dn[id], (float)(xc - x0v));
            if (MODE == 1) acc[0] += wv * yv;
            if (MODE == 3) { acc[0] += (wv - yv) * (wv - yv); acc[1] += wv * wv; }
            if (MODE == 2) { acc[0] += xc * yv; acc[1] += yv * yv; }
            xm = xc;
            xc = xp;
            id += d.plane;
        }
    }
    if (MODE > 0) {
        block_sum<2>(acc, sh);
        if (threadIdx.x == 0 && threadIdx.y == 0) {
            part[blockIdx.x] = acc[0];
            part[RED_MAX_BLOCKS + blockIdx.x] = acc[1];
        }
    }
}

template <int MODE>
__global__ void __launch_bounds__(256) k_helm_km(HelmOp H, const double *__restrict__ x, double *__restrict__ y,
                                                 const double *__restrict__ w, double *part, KTiles t) {
    helm_rows<MODE>(H, x, y, w, part, t, nullptr, nullptr);
}

// residual check of each solve of the set: x = from, A x of the IMMERSED rows
// in `to`; partial sums pstride apart
template <int N>
__global__ void __launch_bounds__(256) k_helm_check(GsSet<N> S, double *part, long pstride, KTiles t) {
    const GsView &V = S.mine();
    helm_rows<3>(V.H, V.from, V.to, V.b, part + (N == 1 ? 0 : blockIdx.y) * pstride, t, V.x0, V.dn);
}

// IMMERSED rows from the sorted IB row table.  With target > 0 each row is
// multiplied by target / (its diagonal): inside the Krylov solve this
// rescales the IB equations (right-hand side 0) to the size of the fluid
// rows, which takes BiCGStab from ~15-20 to 3-4 iterations; any scaled
// residual >= the true one, so the stopping test stays conservative.
__device__ __forceinline__ void ib_apply_row(int a, const long *__restrict__ row, const int *__restrict__ cnt,
                                             const long *__restrict__ col, const double *__restrict__ val,
                                             const double *__restrict__ x, double *__restrict__ y, double target) {
    double s = 0.0, dg = 1.0;
    const long r = row[a];
    const int m = cnt[a];
    // loads first, then the sum in column order (as in k_ib_gs)
    long ci[9];
    double cv[9], xv[9];
#pragma unroll
    for (int e = 0; e < 9; e++) {
        const long ce = e < m ? col[(long)a * 9 + e] : r;
        ci[e] = ce < 0 ? ~ce : ce;
        cv[e] = e < m ? val[(long)a * 9 + e] : 0.0;
    }
#pragma unroll
    for (int e = 0; e < 9; e++) xv[e] = e < m ? x[ci[e]] : 0.0;
#pragma unroll
    for (int e = 0; e < 9; e++) {
        if (e >= m) continue;
        if (ci[e] == r) dg = cv[e];
        s += cv[e] * xv[e];
    }
    double f = (target > 0.0) ? target / dg : 1.0;
    y[r] = (f > 1.0) ? f * s : s;
}

__global__ void k_ib_apply(const long *__restrict__ row, const int *__restrict__ cnt, const long *__restrict__ col,
                           const double *__restrict__ val, int n, const double *__restrict__ x,
                           double *__restrict__ y, double target) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a < n) ib_apply_row(a, row, cnt, col, val, x, y, target);
}

// (A x) of each solve's IMMERSED rows for k_helm_check
template <int N>
__global__ void k_ib_check(GsSet<N> S) {
    const GsView &V = S.mine();
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a < V.nib) ib_apply_row(a, V.row, V.cnt, V.col, V.val, V.from, V.to, 0.0);
}

static HelmOp make_op(tb_ctx *c, int q, double dt) {
    HelmOp H;
    H.d = c->d; H.g = c->g; H.q = q; H.st = c->st[q];
    double kappa = (q == TB_Q_C) ? c->cfg.pe : c->cfg.re;
    H.Cx = -1.0 / (kappa * c->dEta * c->dEta);
    H.Cy = -1.0 / (kappa * c->dXi * c->dXi);
    H.Cz = -1.0 / (kappa * c->dPhi * c->dPhi);
    H.ap_solid = -H.Cx * c->hgrid[15][0] - H.Cy * c->hgrid[16][0] - H.Cz * c->hgrid[17][0];
    H.mod = 1.0 / dt;
    for (int a = 0; a < 6; a++) H.wall[a] = c->cfg.wall_noslip[a];
    H.particle = (q == TB_Q_C && c->cfg.conc_type == TB_PARTICLE);
    H.robin_b_scale = 2.0 / (c->cfg.pe * c->dXi);
    H.vs_abs = fabs(c->cfg.v_settle);
    H.open_w = (q == TB_Q_C) && c->obc.inflow;
    H.open_e = (q != TB_Q_U) && c->obc.outflow;
    return H;
}

// y = A x (scaled: IB rows rescaled for the Krylov solve); mode 1/2 leave
// partial sums in c->red.  Returns the number of partials, or -1.
static int helm_apply(tb_ctx *c, const HelmOp &H, const double *x, double *y, bool scaled, int mode,
                      const double *w = nullptr) {
    int q = H.q;
    if (c->nib[q] > 0)
        hipLaunchKernelGGL(k_ib_apply, dim3((c->nib[q] + 255) / 256), dim3(256), 0, c->s, c->ib_row[q], c->ib_cnt[q],
                           c->ib_col[q], c->ib_val[q], c->nib[q], x, y, scaled ? H.mod : 0.0);
    KTiles t = make_ktiles(c->d.NX, c->d.NY, c->d.NZ);
    if (c->prof_on) tb_prof_begin(c, TB_K_HELM_OP);
    if (mode == 0)
        hipLaunchKernelGGL(k_helm_km<0>, ktiles_grid(t), tiles_block(), 0, c->s, H, x, y, w, c->red, t);
    else if (mode == 1)
        hipLaunchKernelGGL(k_helm_km<1>, ktiles_grid(t), tiles_block(), 0, c->s, H, x, y, w, c->red, t);
    else
        hipLaunchKernelGGL(k_helm_km<2>, ktiles_grid(t), tiles_block(), 0, c->s, H, x, y, w, c->red, t);
    if (c->prof_on) tb_prof_end(c, TB_K_HELM_OP);
    TB_LAUNCH_CHECK(c);
    return (int)(t.per_xcd * NXCD);
}

// ---------------------------------------------------------------------------
// Red-black Gauss-Seidel solve of the Helmholtz system.  The rows are
// dominated by 1/dt (at 512x256x128, Re 2000, dt 1e-3 the off-diagonal sum
// of a fluid row is ~8% of its diagonal), so one red-black sweep reduces the
// error by about two orders of magnitude and a sweep moves ~33 bytes per
// point against ~154 for a BiCGStab iteration.  The solve stops on the same
// test as the reference's KSP, ||b - A x|| <= rtol ||b|| with the true
// residual of the unscaled operator, and hands over to BiCGStab if the
// sweeps stop contracting.

// Per-axis parts of a row, with the terms and wall rules of k_helm_km
// (Velocity.c:449-1471, Conc.c:390-730): d is the axis's share of the
// diagonal with its wall rules folded in, am / ap the minus / plus neighbour
// coefficients (zero where the neighbour is absent).  The diagonal of the
// Gauss-Seidel update is (d_x + d_y) + d_z + 1/dt; it differs from the
// assembled row's only in rounding (the rows sum the same terms in another
// order), so a sweep's fixed point solves the assembled system to ~1e-16.
struct AxisGS {
    double d, am, ap;
};

__device__ inline AxisGS axis_gs(double d, double am, bool hm, int rm, double ap, double wp, bool hp, int rp) {
    AxisGS a;
    if (!hm) d = wallmod(d, am, rm);
    if (!hp) d = wallmod(d, wp, rp);
    a.d = d;
    a.am = hm ? am : 0.0;
    a.ap = hp ? ap : 0.0;
    return a;
}

__device__ inline AxisGS axis_x(const HelmOp &H, int i) {
    const GridDev &g = H.g;
    const int NX = H.d.NX, q = H.q;
    const int *W = H.wall;
    const int im1 = i > 0 ? i - 1 : 0, ip1 = i + 1 < NX ? i + 1 : NX - 1;
    double mpx, mex, mwx;
    if (q == TB_Q_U) { mpx = g.mxu[i]; mex = g.mxc[i]; mwx = g.mxc[im1]; }
    else { mpx = g.mxc[i]; mex = g.mxu[ip1]; mwx = g.mxu[i]; }
    const double Cx = H.Cx;
    const double t = -Cx * mpx * (mex + mwx), aw = Cx * mpx * mwx, ae = Cx * mpx * mex;
    if (q == TB_Q_U) return axis_gs(t, aw, i - 1 >= 1, 0, ae, ae, i + 1 <= NX - 2, 0);
    if (q == TB_Q_C) return axis_gs(t, aw, i > 0, H.open_w ? 0 : 2, ae, ae, i < NX - 2, H.open_e ? 0 : 2);
    return axis_gs(t, aw, i != 0, W[0] ? 1 : 2, ae, ae, i < NX - 2,
                   (i == NX - 2) ? (H.open_e ? 0 : (W[1] ? 1 : 2)) : 0);
}

__device__ inline AxisGS axis_y(const HelmOp &H, int j) {
    const GridDev &g = H.g;
    const int NY = H.d.NY, q = H.q;
    const int *W = H.wall;
    const int jm1 = j > 0 ? j - 1 : 0, jp1 = j + 1 < NY ? j + 1 : NY - 1;
    double mpy, mny, msy;
    if (q == TB_Q_V) { mpy = g.myv[j]; mny = g.myc[j]; msy = g.myc[jm1]; }
    else { mpy = g.myc[j]; mny = g.myv[jp1]; msy = g.myv[j]; }
    const double Cy = H.Cy;
    const double t = -(Cy * mpy * (mny + msy)), as = Cy * mpy * msy, an = Cy * mpy * mny;
    double wn = an;   // top-wall coefficient: the Robin form for settling particles (Conc.c:560-585)
    if (q == TB_Q_C && H.particle) {
        const double bb = H.robin_b_scale * mny;
        wn = an * (bb - H.vs_abs) / (bb + H.vs_abs);
    }
    if (q == TB_Q_V) return axis_gs(t, as, j - 1 >= 1, 0, an, wn, j + 1 <= NY - 2, 0);
    if (q == TB_Q_C) return axis_gs(t, as, j > 0, 2, an, wn, j < NY - 2, 2);
    return axis_gs(t, as, j != 0, W[2] ? 1 : 2, an, wn, j != NY - 2, W[3] ? 1 : 2);
}

__device__ inline AxisGS axis_z(const HelmOp &H, int k) {
    const GridDev &g = H.g;
    const int NZ = H.d.NZ, q = H.q;
    const int *W = H.wall;
    const int km1 = k > 0 ? k - 1 : 0, kp1 = k + 1 < NZ ? k + 1 : NZ - 1;
    double mpz, mbz, mfz;
    if (q == TB_Q_W) { mpz = g.mzw[k]; mbz = g.mzc[km1]; mfz = g.mzc[k]; }
    else { mpz = g.mzc[k]; mbz = g.mzw[k]; mfz = g.mzw[kp1]; }
    const double Cz = H.Cz;
    const double t = -(Cz * mpz * (mbz + mfz)), ab = Cz * mpz * mbz, af = Cz * mpz * mfz;
    if (q == TB_Q_W) return axis_gs(t, ab, k - 1 >= 1, 0, af, af, k + 1 <= NZ - 2, 0);
    if (q == TB_Q_C) return axis_gs(t, ab, k > 0, 2, af, af, k < NZ - 2, 2);
    return axis_gs(t, ab, k != 0, W[4] ? 1 : 2, af, af, k != NZ - 2, W[5] ? 1 : 2);
}

// Gauss-Seidel value of a row of status s from its own current value xp and
// its six neighbour values (clamped to the point itself at the box faces,
// where the coefficient is zero): IMMERSED rows keep xp, other non-fluid
// rows take b / (ap_solid + 1/dt)
__device__ inline double gs_value(const HelmOp &H, const AxisGS &X, const AxisGS &Y, const AxisGS &Z, int s,
                                  double bi, double xp, double xb, double xs, double xw, double xe, double xn,
                                  double xf) {
    const bool fluid = (s == TB_FLUID) || (H.q != TB_Q_C && s == TB_BUFFER_SOLID);
    double o = Z.am * xb;
    o = fma(Y.am, xs, o);
    o = fma(X.am, xw, o);
    o = fma(X.ap, xe, o);
    o = fma(Y.ap, xn, o);
    o = fma(Z.ap, xf, o);
    const double num = fluid ? bi - o : bi;
    const double den = fluid ? ((X.d + Y.d) + Z.d) + H.mod : H.ap_solid + H.mod;
    const double v = num / den;
    return s == TB_IMMERSED ? xp : v;
}

// One red-black sweep pair over the non-IMMERSED rows in a single pass:
// xn = black(red(xo)), red = (i + j + k) even, updated first.  Every red
// value reads only black neighbours of xo and every black value only red
// neighbours of the red pass (a neighbour clamped to the point itself reads
// the point's own current value), so the pair is the same iteration as two
// in-place colour passes (equal to rounding: the diagonals are summed per
// axis, see AxisGS), while xo and b are read from HBM once and xn written
// once (the in-place form streams both arrays twice).
//
// A 512-thread block owns a 64 x 16 column tile and a chunk of T.tk planes
// and walks k upwards through two LDS rings: four planes of xo with a
// two-point halo, and three of the red-pass values (black positions holding
// xo) with a one-point halo.  Per plane m, with two barriers: store plane m-2
// (both of its passes are done) and red pass on plane m (tile + halo,
// recomputed by the neighbouring tiles); black pass on plane m-1 (tile).
// The fourth xo plane lets the next plane's staging overlap the black pass.
// The chunk recomputes the red pass on one plane below and above.  The
// xo plane, statuses and right-hand sides of the next plane are fetched into
// registers one step ahead, so their latency overlaps the passes; row
// coefficients come from per-axis tables built in LDS once per block.
// Chunks of up to 32 planes: a block is a chain of tk + 3 plane steps behind
// a start of about three more, and 512 blocks are resident at once (two per
// CU at 75 KB of LDS; two of a CU take 8/5 of the time per step that one does:
// 2.9 against 1.8 us), so make_gs_tiles takes the chunk with the least time in
// sequence.  At 512 x 256 x 128 that is 32 (8 x 16 x 4 tiles, one round;
// 126 -> 115 us per pair against 16 planes); small grids fill the chip with
// short chains instead of leaving most of it idle (64 -> 11 us a pair at
// 128x64x32).
constexpr int GS_TX = 64, GS_TY = 16, GS_TK_MAX = 32;
constexpr int GS_OX = GS_TX + 4, GS_OY = GS_TY + 4;   // xo ring: halo 2
constexpr int GS_HX = GS_TX + 2, GS_HY = GS_TY + 2;   // red-pass ring: halo 1
constexpr int GS_OZ = GS_TK_MAX + 4;                  // z table: k0-2 .. k0+tk+1
constexpr int GS_ORING = 4;                           // xo planes staged: m-1, m, m+1 and the next
constexpr int GS_THREADS = 512;
constexpr int GS_OLD_PER = (GS_OY * GS_OX + GS_THREADS - 1) / GS_THREADS;
constexpr int GS_RED = GS_HY * (GS_HX / 2);           // red points of one halo plane
constexpr int GS_RED_PER = (GS_RED + GS_THREADS - 1) / GS_THREADS;
static_assert(GS_TX * GS_TY == 2 * GS_THREADS, "one black point per thread");
static_assert(GS_TX % 2 == 0, "tile origins must be even");

struct GsTiles {
    int tx, ty, kc, tk;   // tiles per axis, planes per chunk
    int n, per_xcd;
};

constexpr long GS_RESIDENT = 512;   // blocks resident at once
constexpr int GS_START = 3;         // plane steps a block's start takes

// The tiles cover the box without its last plane along each axis (see
// k_gs_last_planes), so 512 x 256 x 128 cells take exactly 8 x 16 x 4 tiles
// instead of 9 x 17 x 9 with nearly empty ones walking the full plane chain.
// nq: solves in the launch
static GsTiles make_gs_tiles(const Dims &d, int nq) {
    GsTiles t;
    t.tx = (d.NX - 1 + GS_TX - 1) / GS_TX;
    t.ty = (d.NY - 1 + GS_TY - 1) / GS_TY;
    long best = 0;
    for (int tk = GS_TK_MAX; tk >= 1; tk--) {
        const long kc = (d.NZ - 1 + tk - 1) / tk, n = t.tx * t.ty * kc * nq;
        const long step = n <= GS_RESIDENT / 2 ? 5 : 8 * ((n + GS_RESIDENT - 1) / GS_RESIDENT);
        const long cost = step * (tk + 3 + GS_START);
        if (best == 0 || cost < best) { best = cost; t.tk = tk; t.kc = (int)kc; }
    }
    t.n = t.tx * t.ty * t.kc;
    t.per_xcd = (t.n + NXCD - 1) / NXCD;
    return t;
}

// Neighbours are read without clamping at the box faces: every row whose
// neighbour index leaves the box either has a zero coefficient there or is
// not a FLUID row (the last plane of each axis is BOUNDARY), and the LDS
// positions outside the box hold zeros or finite values of other planes.
// Element offsets are 32-bit (the host checks the field size).  ADD: the
// pair starts from xo + dd (the field plus the last solve's increment, an
// extrapolated initial guess; dd null: xo) without forming it in memory.
template <bool ADD>
__device__ __forceinline__ void gs_pair(const HelmOp &H, const double *__restrict__ xo, double *__restrict__ xn,
                                        const double *__restrict__ b, const GsTiles &T,
                                        const float *__restrict__ dd) {
    __shared__ double so[GS_ORING][GS_OY * GS_OX];
    __shared__ double sr[3][GS_HY * GS_HX];
    __shared__ AxisGS cx[GS_OX], cy[GS_OY], cz[GS_OZ];
    const Dims &d = H.d;
    const int NX = d.NX, NY = d.NY, NZ = d.NZ, px = d.px;
    const int plane = (int)d.plane;
    const int bid = blockIdx.x;
    const int lt = (bid % NXCD) * T.per_xcd + bid / NXCD;   // consecutive tiles share an XCD's L2
    if (lt >= T.n) return;                                  // whole block
    const int tx = lt % T.tx, rest = lt / T.tx;
    const int i0 = tx * GS_TX, j0 = (rest % T.ty) * GS_TY;
    const int k0 = (rest / T.ty) * T.tk;
    const int k1 = k0 + T.tk < NZ - 1 ? k0 + T.tk : NZ - 1;   // the last plane: k_gs_last_planes
    const int t = threadIdx.x;
    const uint8_t *__restrict__ st = H.st;

    for (int e = t; e < GS_ORING * GS_OY * GS_OX; e += GS_THREADS) (&so[0][0])[e] = 0.0;
    for (int e = t; e < 3 * GS_HY * GS_HX; e += GS_THREADS) (&sr[0][0])[e] = 0.0;
    for (int e = t; e < GS_OX + GS_OY + GS_OZ; e += GS_THREADS) {
        if (e < GS_OX) {
            const int i = i0 - 2 + e;
            if (i >= 0 && i < NX) cx[e] = axis_x(H, i);
        } else if (e < GS_OX + GS_OY) {
            const int j = j0 - 2 + (e - GS_OX);
            if (j >= 0 && j < NY) cy[e - GS_OX] = axis_y(H, j);
        } else {
            const int k = k0 - 2 + (e - GS_OX - GS_OY);
            if (k >= 0 && k < NZ) cz[e - GS_OX - GS_OY] = axis_z(H, k);
        }
    }
    __syncthreads();   // zeros in place before the first planes are staged

    // xo plane staging: in-plane offset of each of this thread's halo-2
    // points (-1 outside the box); the LDS index is e itself
    int ooff[GS_OLD_PER];
#pragma unroll
    for (int u = 0; u < GS_OLD_PER; u++) {
        const int e = t + u * GS_THREADS;
        const int r = e / GS_OX, cc = e - r * GS_OX;
        const int i = i0 - 2 + cc, j = j0 - 2 + r;
        ooff[u] = (e < GS_OY * GS_OX && i >= 0 && i < NX && j >= 0 && j < NY) ? j * px + i : -1;
    }
    // the loads of a plane stay in flight until put_old (with ADD the sum is
    // formed there too, not between the loads)
    double ro[GS_OLD_PER];
    float rd[GS_OLD_PER];   // widened where the sum is formed, so the load is not waited for here
    auto fetch_old = [&](int m) {
#pragma unroll
        for (int u = 0; u < GS_OLD_PER; u++) {
            ro[u] = ooff[u] >= 0 ? xo[m * plane + ooff[u]] : 0.0;
            if (ADD) rd[u] = dd && ooff[u] >= 0 ? dd[m * plane + ooff[u]] : 0.0f;
        }
    };
    auto put_old = [&](int m) {
        double *S = so[m % GS_ORING];
#pragma unroll
        for (int u = 0; u < GS_OLD_PER; u++) {
            const int e = t + u * GS_THREADS;
            if (e < GS_OY * GS_OX) S[e] = ADD ? ro[u] + (double)rd[u] : ro[u];
        }
    };
    // this thread's red points of the halo-1 plane: row, column pair, y
    int rrow[GS_RED_PER], rc2[GS_RED_PER];
#pragma unroll
    for (int u = 0; u < GS_RED_PER; u++) {
        const int e = t + u * GS_THREADS;
        rrow[u] = e < GS_RED ? e / (GS_HX / 2) : 0;
        rc2[u] = e < GS_RED ? e - rrow[u] * (GS_HX / 2) : -1;
    }
    // status (-1 outside the box) and b of the red points of plane m
    int rs[GS_RED_PER];
    double rb[GS_RED_PER];
    auto fetch_red = [&](int m, int *s_, double *b_) {
#pragma unroll
        for (int u = 0; u < GS_RED_PER; u++) {
            const int j = j0 - 1 + rrow[u];
            const int i = i0 - 1 + 2 * rc2[u] + ((1 + j + m) & 1);   // i + j + m even (i0 is even)
            s_[u] = -1;
            b_[u] = 0.0;
            if (rc2[u] >= 0 && i >= 0 && i < NX && j >= 0 && j < NY) {
                const int id = m * plane + j * px + i;
                s_[u] = st[id];
                b_[u] = b[id];
            }
        }
    };
#pragma unroll
    for (int u = 0; u < GS_RED_PER; u++) { rs[u] = -1; rb[u] = 0.0; }
    // this thread's black point of plane k
    const int br = t / (GS_TX / 2), bc2 = t % (GS_TX / 2);
    const int bj = j0 + br;
    int bs = -1;
    double bbv = 0.0;
    auto fetch_black = [&](int k, int &s_, double &b_) {
        const int i = i0 + 2 * bc2 + ((1 + bj + k) & 1);
        s_ = -1;
        b_ = 0.0;
        if (i < NX && bj < NY) {
            const int id = k * plane + bj * px + i;
            s_ = st[id];
            b_ = b[id];
        }
    };

    // both colours of plane k, from its sr slot to xn (coalesced rows)
    auto write_plane = [&](int k) {
        if (k < k0 || k >= k1) return;
        const double *R = sr[k % 3];
        for (int e = t; e < GS_TY * GS_TX; e += GS_THREADS) {
            const int r = e / GS_TX, cc = e - r * GS_TX;
            const int i = i0 + cc, j = j0 + r;
            if (i < NX && j < NY) st_stream(&xn[k * plane + j * px + i], R[(r + 1) * GS_HX + cc + 1]);
        }
    };

    if (k0 >= 2) { fetch_old(k0 - 2); put_old(k0 - 2); }
    if (k0 >= 1) { fetch_old(k0 - 1); put_old(k0 - 1); }
    fetch_old(k0);
    if (k0 >= 1) fetch_red(k0 - 1, rs, rb);
    for (int m = k0 - 1; m <= k1; m++) {
        if (m + 1 < NZ) put_old(m + 1);
        if (m + 2 < NZ) fetch_old(m + 2);
        int rs_n[GS_RED_PER];
        double rb_n[GS_RED_PER];
#pragma unroll
        for (int u = 0; u < GS_RED_PER; u++) { rs_n[u] = -1; rb_n[u] = 0.0; }
        if (m + 1 < NZ) fetch_red(m + 1, rs_n, rb_n);
        int bs_n = -1;
        double bb_n = 0.0;
        if (m >= k0 && m < k1) fetch_black(m, bs_n, bb_n);
        __syncthreads();
        // plane m - 2 is final (its black pass ran in the previous
        // iteration) and its sr slot is next written by the red pass of m + 1
        write_plane(m - 2);
        if (m >= 0 && m < NZ) {
            // red pass on plane m over the tile + halo 1
            const double *S = so[m % GS_ORING], *Sb = so[(m + GS_ORING - 1) % GS_ORING],
                         *Sf = so[(m + 1) % GS_ORING];
            double *R = sr[m % 3];
            const AxisGS Z = cz[m - k0 + 2];
#pragma unroll
            for (int u = 0; u < GS_RED_PER; u++) {
                const int s = rs[u];
                if (s < 0) continue;
                const int r = rrow[u];
                const int cc = 2 * rc2[u] + ((j0 + r + m) & 1);
                const int o = (r + 1) * GS_OX + cc + 1;
                R[r * GS_HX + cc] = gs_value(H, cx[cc + 1], cy[r + 1], Z, s, rb[u], S[o], Sb[o], S[o - GS_OX],
                                             S[o - 1], S[o + 1], S[o + GS_OX], Sf[o]);
            }
        }
        __syncthreads();
        const int k = m - 1;
        if (k >= k0 && k < k1 && bs >= 0) {
            // black pass on plane k over the tile, into the black positions of sr
            double *R = sr[k % 3];
            const double *Rb = sr[(k + 2) % 3], *Rf = sr[(k + 1) % 3];
            const int cc = 2 * bc2 + ((1 + bj + k) & 1);
            const int h = (br + 1) * GS_HX + cc + 1;
            R[h] = gs_value(H, cx[cc + 2], cy[br + 2], cz[k - k0 + 2], bs, bbv,
                            so[k % GS_ORING][(br + 2) * GS_OX + cc + 2], Rb[h], R[h - GS_HX], R[h - 1], R[h + 1],
                            R[h + GS_HX], Rf[h]);
        }
        // no barrier here: the next iteration's staging writes the xo slot of
        // plane m + 2, which no pass of this iteration reads (GS_ORING = 4),
        // and its first barrier precedes every read of this black pass
#pragma unroll
        for (int u = 0; u < GS_RED_PER; u++) { rs[u] = rs_n[u]; rb[u] = rb_n[u]; }
        bs = bs_n;
        bbv = bb_n;
    }
    __syncthreads();
    write_plane(k1 - 1);
}

template <bool ADD, int N>
__global__ void __launch_bounds__(GS_THREADS) k_helm_gs_pair(GsSet<N> S, GsTiles T) {
    const GsView &V = S.mine();
    gs_pair<ADD>(V.H, V.from, V.to, V.b, T, V.inc);
}

// The last plane of each axis, outside the sweep tiles.  Its points are
// BOUNDARY by classification: their rows read ap_solid q = b and no other
// row couples to them (zero coefficients), so their Gauss-Seidel value
// b / (ap_solid + 1/dt), the expression of gs_value, does not depend on x and
// is written into both iterate buffers (from and to) once per solve.  Points
// where two planes meet are written twice with the same value.
template <int N>
__global__ void k_gs_last_planes(GsSet<N> S) {
    const GsView &V = S.mine();
    const HelmOp &H = V.H;
    const double *b = V.b;
    double *x1 = const_cast<double *>(V.from), *x2 = V.to;
    const Dims &d = H.d;
    const long n1 = (long)d.NY * d.NZ, n2 = (long)d.NX * d.NZ, n3 = (long)d.NX * d.NY;
    long e = blockIdx.x * (long)blockDim.x + threadIdx.x;
    int i, j, k;
    if (e < n1) {
        i = d.NX - 1; j = (int)(e % d.NY); k = (int)(e / d.NY);
    } else if ((e -= n1) < n2) {
        j = d.NY - 1; i = (int)(e % d.NX); k = (int)(e / d.NX);
    } else if ((e -= n2) < n3) {
        k = d.NZ - 1; i = (int)(e % d.NX); j = (int)(e / d.NX);
    } else {
        return;
    }
    const long id = gidx(d, i, j, k);
    if (H.st[id] == TB_IMMERSED) return;   // kept, as the sweep keeps IMMERSED rows
    const double v = b[id] / (H.ap_solid + H.mod);
    x1[id] = v;
    x2[id] = v;
}

// IMMERSED rows, Jacobi over the IB table (x_im = (b_im - sum_{g != im} v_g
// x_g) / v_im): the row's new value is written over the old one that the pair
// left in `to`; other IMMERSED nodes (complemented columns) are read where the
// pair read them, in `from` (+ inc), so the result does not depend on the
// order in which rows run and takes one launch (with a buffer between and a
// second one it was 4 + 3 us and a gap at 200x72x36, 8 + 5 at 512x256x128).
template <int N>
__global__ void k_ib_gs(GsSet<N> S) {
    const GsView &V = S.mine();
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= V.nib) return;
    const double *from = V.from, *b = V.b;
    double *x = V.to;
    const float *inc = V.inc;
    const long r = V.row[a];
    const int m = V.cnt[a];
    // every column and value, then every gather, issued before the first
    // is used; the sum runs in column order as a loop over them would
    long ci[9];
    double cv[9], xv[9];
#pragma unroll
    for (int e = 0; e < 9; e++) {
        ci[e] = e < m ? V.col[(long)a * 9 + e] : r;
        cv[e] = e < m ? V.val[(long)a * 9 + e] : 0.0;
    }
#pragma unroll
    for (int e = 0; e < 9; e++) {
        xv[e] = 0.0;
        if (e >= m || ci[e] == r) continue;
        if (ci[e] >= 0) xv[e] = x[ci[e]];
        else xv[e] = inc ? from[~ci[e]] + (double)inc[~ci[e]] : from[~ci[e]];
    }
    double s = 0.0, dg = 1.0;
#pragma unroll
    for (int e = 0; e < 9; e++) {
        if (e >= m) continue;
        if (ci[e] == r) dg = cv[e];
        else s += cv[e] * xv[e];
    }
    x[r] = (b[r] - s) / dg;
}

// One quantity's Gauss-Seidel solve
struct GsRun {
    int q = 0;
    int field = 0;                 // concentration field (q = TB_Q_C)
    HelmOp H;
    double *x = nullptr;           // the field; kept while the solve runs
    const double *b = nullptr;
    double *cur = nullptr, *alt = nullptr;   // iterate buffers
    bool spare = false;            // alt comes from the history's third buffer, else kv[6]
    const double *src = nullptr;   // start of the first pair (else cur)
    const float *inc = nullptr;    // and the increment added to it
    bool planes = false;           // last planes written
    HelmHistory h;
    int nib = 0;
    const long *row = nullptr, *col = nullptr;
    const int *cnt = nullptr;
    const double *val = nullptr;
    int par = 0, chunk = 0, todo = 0, its = 0;
    double prev = NAN, rate = 0.0, res = NAN;
    bool done = false, ok = false;
};

static void gs_ib(tb_ctx *c, GsRun &r) {
    const int q = r.q;
    r.nib = c->nib[q];
    r.row = c->ib_row[q]; r.col = c->ib_col[q]; r.cnt = c->ib_cnt[q]; r.val = c->ib_val[q];
}

static GsView view(const GsRun &r, const double *from, double *to, const float *inc) {
    return {r.H, r.b, r.x, from, to, inc, r.h.inc, r.row, r.col, r.cnt, r.val, r.nib};
}

// up to todo sweep pairs of each run, each followed by the Jacobi update of
// the IMMERSED rows, alternating between the buffers cur and alt (the same
// size and pitch); cur is swapped to the buffer that holds the result
template <int N>
static int gs_pairs(tb_ctx *c, GsRun *const *run, int n) {
    if (c->d.ntot >= (1L << 31)) {
        c->err = "Helmholtz sweeps: field exceeds 2^31 elements";
        return -1;
    }
    const Dims &d = c->d;
    GsSet<N> S;
    int m = 0, most = 0;
    for (int a = 0; a < n; a++) {
        most = run[a]->todo > most ? run[a]->todo : most;
        if (run[a]->planes || run[a]->todo < 1) continue;
        run[a]->planes = true;
        S.v[m++] = view(*run[a], run[a]->cur, run[a]->alt, nullptr);
    }
    if (m > 0) {
        const long np = (long)d.NY * d.NZ + (long)d.NX * d.NZ + (long)d.NX * d.NY;
        hipLaunchKernelGGL(k_gs_last_planes<N>, dim3((unsigned)((np + 255) / 256), m), dim3(256), 0, c->s, S);
        TB_LAUNCH_CHECK(c);
    }
    for (int sw = 0; sw < most; sw++) {
        int nib = 0;
        bool add = false;
        m = 0;
        for (int a = 0; a < n; a++) {
            GsRun &r = *run[a];
            if (sw >= r.todo) continue;
            S.v[m++] = view(r, r.src ? r.src : r.cur, r.alt, r.src ? r.inc : nullptr);
            add |= r.src && r.inc;
            nib = r.nib > nib ? r.nib : nib;
            r.src = nullptr;
            std::swap(r.cur, r.alt);
        }
        const GsTiles T = make_gs_tiles(d, m);
        const dim3 grid(T.per_xcd * NXCD, m);
        if (add) TB_PROF(c, TB_K_HELM_GS, hipLaunchKernelGGL((k_helm_gs_pair<true, N>), grid, dim3(GS_THREADS), 0, c->s, S, T));
        else TB_PROF(c, TB_K_HELM_GS, hipLaunchKernelGGL((k_helm_gs_pair<false, N>), grid, dim3(GS_THREADS), 0, c->s, S, T));
        if (nib > 0)
            TB_PROF(c, TB_K_IB, hipLaunchKernelGGL(k_ib_gs<N>, dim3((nib + 255) / 256, m), dim3(256), 0, c->s, S));
        TB_LAUNCH_CHECK(c);
    }
    return 0;
}

// |b - A x|^2 and |b|^2 of each run's iterate into hscal[S_SUB + 2 a ...], its
// increment over the field into h.inc; the other iterate's IMMERSED rows,
// which no pair reads, hold A x in between
template <int N>
static int gs_check(tb_ctx *c, GsRun *const *run, int n) {
    constexpr long PART = RED_MAX_BLOCKS / HELM_SET;
    GsSet<N> S;
    int nib = 0;
    for (int a = 0; a < n; a++) {
        S.v[a] = view(*run[a], run[a]->cur, run[a]->alt, nullptr);
        nib = run[a]->nib > nib ? run[a]->nib : nib;
    }
    if (nib > 0) hipLaunchKernelGGL(k_ib_check<N>, dim3((nib + 255) / 256, n), dim3(256), 0, c->s, S);
    const KTiles t = make_ktiles(c->d.NX, c->d.NY, c->d.NZ, true);
    dim3 grid = ktiles_grid(t);
    grid.y = n;
    TB_PROF(c, TB_K_HELM_OP, hipLaunchKernelGGL(k_helm_check<N>, grid, tiles_block(), 0, c->s, S, c->red, PART, t));
    TB_LAUNCH_CHECK(c);
    TB_CHECK(c, hipEventRecord(c->ev1, c->s));   // the sums below end after it
    return tb_reduce_read(c, (int)(t.per_xcd * NXCD), 2, S_SUB, n, PART);
}

// copy the box points of src into dst (row padding untouched)
static int copy_box(tb_ctx *c, double *dst, const double *src) {
    const size_t pitch = sizeof(double) * (size_t)c->d.px;
    TB_CHECK(c, hipMemcpy2DAsync(dst, pitch, src, pitch, sizeof(double) * (size_t)c->d.NX,
                                 (size_t)c->d.NY * c->d.NZ, hipMemcpyDeviceToDevice, c->s));
    return 0;
}

// Grids up to this size have all their quantities solved as one set, each with
// a third iterate buffer of its own.  Four quantities' solves of a step, one by
// one and as a set: 0.59 and 0.24 ms at 64x16x16, 1.00 / 0.58 at 192x64x64,
// 1.59 / 0.86 at 256x128x64, 3.37 / 2.93 at 512x128x128 and 6.87 / 6.58 at
// 512x256x128, where a launch's last round of blocks is what is left to share;
// beyond, that is not worth the memory.
constexpr long HELM_SET_POINTS = 1L << 25;

// the run of quantity q (the selected concentration field's for TB_Q_C)
static int gs_begin(tb_ctx *c, int q, const HelmOp &H, bool spare, GsRun &r) {
    if (tb_helm_inc_alloc(c, q)) return -1;
    r.spare = spare;
    r.q = q;
    r.field = c->conc_sel;
    r.H = H;
    r.x = c->f[TB_F_U + q];
    r.b = c->f[TB_F_RHS_U + q];
    r.h = c->helm[q];
    gs_ib(c, r);
    r.src = r.x;
    r.inc = r.h.inc_ok ? r.h.inc : nullptr;
    c->helm[q].inc_ok = r.h.inc_ok = false;   // the increment is overwritten by the first residual check
    r.cur = r.h.buf;
    r.alt = r.spare ? r.h.spare : c->kv[6];
    r.par = (int)(r.h.nsolve++ & 1u);
    r.chunk = r.h.sweeps[r.par] > 0 ? r.h.sweeps[r.par] : 2;
    r.rate = r.h.rate[r.par];
    return 0;
}

// sets ok of the runs that converged; the others stalled (contraction per
// pair worse than 0.5) or ran out of sweeps, cur then holds the last iterate.
// The initial guess is the field plus the increment of the quantity's last
// solve, when that solve converged on the same trajectory (the reference
// starts from the field alone; both stop at the same residual test).  Three
// FP64 buffers take part: the field x, read by the first pair and kept so
// that each residual check also writes the increment, and the two iterate
// buffers, the quantity's second buffer and its third (in a set) or kv[6].
// The increment is kept in FP32: it only moves the start of the next solve,
// which converges to the same residual test, and the check that writes it
// and the first pair that reads it stream half the bytes for it.
// The true residual costs about two thirds of a sweep pair, so it is
// evaluated only where the solve may have converged: first after as many
// pairs as the last solve of the same quantity and RK stage parity needed
// (the count is steady from step to step), then after the pairs predicted
// from the observed contraction (at most 3 at a time: the contraction
// improves as the sweeps go, a longer prediction overshoots).  The initial
// residual is not evaluated (res0 = NaN).
template <int N>
static int gs_solve(tb_ctx *c, GsRun *run, int n, double rtol, int maxit) {
    for (;;) {
        GsRun *act[N];
        int m = 0;
        for (int a = 0; a < n; a++) {
            GsRun &r = run[a];
            if (r.done || r.its >= maxit) continue;
            r.todo = r.chunk < maxit - r.its ? r.chunk : maxit - r.its;
            act[m++] = &r;
        }
        if (m == 0) break;
        if (gs_pairs<N>(c, act, m) || gs_check<N>(c, act, m)) return -1;
        for (int a = 0; a < m; a++) {
            GsRun &r = *act[a];
            const double rr = c->hscal[S_SUB + 2 * a], bb = c->hscal[S_SUB + 2 * a + 1];
            double bn = sqrt(bb);
            if (bn == 0.0) bn = 1.0;
            r.its += r.todo;
            r.res = sqrt(rr) / bn;
            r.ok = r.res <= rtol;
            r.done = r.ok || !(r.res == r.res);
            if (r.done) continue;
            if (r.prev == r.prev) r.rate = pow(r.res / r.prev, 1.0 / r.todo);
            r.prev = r.res;
            if (!(r.rate > 0.0)) r.rate = 0.05;   // no estimate yet
            if (!(r.rate < 0.5)) { r.done = true; continue; }
            const int need = (int)ceil(log(rtol / r.res) / log(r.rate));
            r.chunk = need < 1 ? 1 : (need > 3 ? 3 : need);
        }
    }
    for (int a = 0; a < n; a++) {
        GsRun &r = run[a];
        if (!r.ok) continue;
        // one pair fewer next time when this residual shows it would have
        // sufficed at the last contraction
        const double r1 = (r.rate > 0.0 && r.rate < 0.5) ? r.rate : 0.05;
        r.h.sweeps[r.par] = (r.its > 1 && r.res / r1 <= rtol) ? r.its - 1 : r.its;
        if (r.prev == r.prev) r.h.rate[r.par] = r.rate;
    }
    return 0;
}

// The run's result into the context (with its concentration field selected):
// the field takes the result's buffer, the second buffer the other
// iterate's and the third one (or kv[6]) the old field's (no kernel or graph
// keeps any of these pointers between calls).
static int gs_end(tb_ctx *c, GsRun &r) {
    const int q = r.q;
    c->helm[q] = r.h;
    if (!r.ok) return copy_box(c, r.x, r.cur);   // BiCGStab continues from x
    c->f[TB_F_U + q] = r.cur;
    c->helm[q].buf = r.alt;
    if (r.spare) c->helm[q].spare = r.x;
    else c->kv[6] = r.x;
    c->helm[q].inc_ok = true;
    return 0;
}

static void gs_stats(const GsRun &r, double ms, tb_solve_stats *st) {
    if (!st) return;
    st->iterations = r.its;
    st->converged = 1;
    st->fallback = 0;
    st->vcycles = 0;
    st->res0 = NAN;
    st->res = r.res;
    st->ms = ms;
}

// The smoother of tb_helmholtz_solve by itself: f_x <- `pairs` red-black
// sweep pairs (each followed by the Jacobi update of the IMMERSED rows) of
// A_q(dt) x = f_b, in place.
extern "C" int tb_helmholtz_gs_sweeps(tb_ctx *c, int q, double dt, int f_b, int f_x, int pairs) {
    if (!c || q < 0 || q > 3 || f_b < 0 || f_b >= TB_F_COUNT || f_x < 0 || f_x >= TB_F_COUNT || f_b == f_x ||
        pairs < 0) {
        if (c) c->err = "tb_helmholtz_gs_sweeps: bad argument";
        return -1;
    }
    tb_field_written(c, f_x);
    GsRun r, *one = &r;
    r.q = q;
    r.H = make_op(c, q, dt);
    r.b = c->f[f_b];
    gs_ib(c, r);
    r.cur = c->f[f_x];
    r.alt = c->kv[6];
    r.todo = pairs;
    if (gs_pairs<1>(c, &one, 1)) return -1;
    if (r.cur != c->f[f_x] && copy_box(c, c->f[f_x], r.cur)) return -1;
    TB_CHECK(c, hipStreamSynchronize(c->s));
    return 0;
}

extern "C" int tb_helmholtz_apply(tb_ctx *c, int q, double dt, int f_in, int f_out) {
    if (!c || q < 0 || q > 3 || f_in < 0 || f_in >= TB_F_COUNT || f_out < 0 || f_out >= TB_F_COUNT || f_in == f_out) {
        if (c) c->err = "tb_helmholtz_apply: bad argument";
        return -1;
    }
    tb_field_written(c, f_out);
    HelmOp H = make_op(c, q, dt);
    if (helm_apply(c, H, c->f[f_in], c->f[f_out], false, 0) < 0) return -1;
    TB_CHECK(c, hipStreamSynchronize(c->s));
    return 0;
}

// ---------------------------------------------------------------------------
// vector kernels with reductions (partials in c->red, RED_MAX_BLOCKS apart)

constexpr int VB = 1024;   // blocks of the grid-stride vector kernels
constexpr int VT = 256;

// r = b - y ; rhat = r ; p = v = 0 ; partials: r.r, b.b
__global__ void k_bicg_init(long n, const double *__restrict__ b, const double *__restrict__ y,
                            double *__restrict__ r, double *__restrict__ rh, double *__restrict__ p,
                            double *__restrict__ v, double *part) {
    __shared__ double sh[32];
    double acc[2] = {0.0, 0.0};
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        double bi = b[i];
        double ri = bi - y[i];
        r[i] = ri; rh[i] = ri; p[i] = 0.0; v[i] = 0.0;
        acc[0] += ri * ri;
        acc[1] += bi * bi;
    }
    block_sum<2>(acc, sh);
    if (threadIdx.x == 0) { part[blockIdx.x] = acc[0]; part[RED_MAX_BLOCKS + blockIdx.x] = acc[1]; }
}

// scalar updates on the device
__global__ void k_scalar(double *s, int op) {
    if (threadIdx.x != 0) return;
    switch (op) {
    case 0:   // start: rho = alpha = omega = 1
        s[S_RHO] = 1.0; s[S_ALPHA] = 1.0; s[S_OMEGA] = 1.0;
        break;
    case 1: { // beta = (rho1/rho)*(alpha/omega) ; rho = rho1 (rho1 in S_RHV)
        double rho1 = s[S_RHV];
        s[S_BETA] = (rho1 / s[S_RHO]) * (s[S_ALPHA] / s[S_OMEGA]);
        s[S_RHO] = rho1;
        break;
    }
    case 2:   // alpha = rho / (rhat.v) (in S_TMP0)
        s[S_ALPHA] = s[S_RHO] / s[S_TMP0];
        break;
    case 3:   // omega = (t.s)/(t.t)
        s[S_OMEGA] = (s[S_TT] > 0.0) ? s[S_TS] / s[S_TT] : 0.0;
        break;
    }
}

__global__ void k_bicg_p(long n, const double *__restrict__ r, const double *__restrict__ v, double *__restrict__ p,
                         const double *__restrict__ s) {
    double beta = s[S_BETA], omega = s[S_OMEGA];
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        p[i] = r[i] + beta * (p[i] - omega * v[i]);
}

__global__ void k_bicg_s(long n, const double *__restrict__ r, const double *__restrict__ v, double *__restrict__ sv,
                         const double *__restrict__ s) {
    double alpha = s[S_ALPHA];
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        sv[i] = r[i] - alpha * v[i];
}

// x += alpha p + omega s ; r = s - omega t ; partials r.r and rhat.r
__global__ void k_bicg_xr(long n, double *__restrict__ x, double *__restrict__ r, const double *__restrict__ p,
                          const double *__restrict__ sv, const double *__restrict__ t, const double *__restrict__ rh,
                          const double *__restrict__ s, double *part) {
    __shared__ double sh[32];
    double alpha = s[S_ALPHA], omega = s[S_OMEGA];
    double acc[2] = {0.0, 0.0};
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        double si = sv[i];
        x[i] += alpha * p[i] + omega * si;
        double ri = si - omega * t[i];
        r[i] = ri;
        acc[0] += ri * ri;
        acc[1] += rh[i] * ri;
    }
    block_sum<2>(acc, sh);
    if (threadIdx.x == 0) { part[blockIdx.x] = acc[0]; part[RED_MAX_BLOCKS + blockIdx.x] = acc[1]; }
}

__global__ void k_sub(long n, const double *__restrict__ b, const double *__restrict__ y, double *__restrict__ r,
                      double *part) {
    __shared__ double sh[16];
    double acc[1] = {0.0};
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        double ri = b[i] - y[i];
        r[i] = ri;
        acc[0] += ri * ri;
    }
    block_sum<1>(acc, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = acc[0];
}

__global__ void k_copy_slot(double *s, int dst, int src) {
    if (threadIdx.x == 0) s[dst] = s[src];
}

static int read_scalars(tb_ctx *c, int first, int count) { return tb_read_scalars(c, first, count); }

// BiCGStab (van der Vorst 1992), the method of KSPIBCGS (Solver.c:39-86,
// 269-322), with the IB equations rescaled (see k_ib_apply); nonzero initial
// guess = the current field; stops at ||b - A x|| <= rtol ||b|| (PETSc's
// default test relative to the right-hand side), checked on the true
// residual at the end.
// handover: 1 when the Gauss-Seidel sweeps stopped contracting (or ran out of
// pairs) and this finishes the solve.
static int bicgstab(tb_ctx *c, int q, const HelmOp &H, int handover, tb_solve_stats *st) {
    long n = c->d.ntot;
    double *x = c->f[TB_F_U + q], *b = c->f[TB_F_RHS_U + q];
    double *r = c->kv[0], *rh = c->kv[1], *p = c->kv[2], *v = c->kv[3], *sv = c->kv[4], *t = c->kv[5];
    const double rtol = c->cfg.helm_rtol;
    const int maxit = c->cfg.helm_maxit;
    c->helm[q].inc_ok = false;   // the increment is recorded by the Gauss-Seidel solve only
    if (helm_apply(c, H, x, t, true, 0) < 0) return -1;
    hipLaunchKernelGGL(k_bicg_init, dim3(VB), dim3(VT), 0, c->s, n, b, t, r, rh, p, v, c->red);
    if (tb_reduce_finish(c, VB, 2, S_RR)) return -1;   // S_RR = r.r, S_RR+1 = b.b
    hipLaunchKernelGGL(k_scalar, dim3(1), dim3(64), 0, c->s, c->scal, 0);
    TB_LAUNCH_CHECK(c);
    if (read_scalars(c, S_RR, 2)) return -1;
    double rr = c->hscal[S_RR], bb = c->hscal[S_RR + 1];
    double bn = sqrt(bb);
    if (bn == 0.0) bn = 1.0;
    double res0 = sqrt(rr) / bn, res = res0;
    hipLaunchKernelGGL(k_copy_slot, dim3(1), dim3(64), 0, c->s, c->scal, S_RHV, S_RR);   // rhat.r = r.r
    int it = 0;
    bool conv = res <= rtol;
    while (!conv && it < maxit) {
        hipLaunchKernelGGL(k_scalar, dim3(1), dim3(64), 0, c->s, c->scal, 1);
        hipLaunchKernelGGL(k_bicg_p, dim3(VB), dim3(VT), 0, c->s, n, r, v, p, c->scal);
        int nb = helm_apply(c, H, p, v, true, 1, rh);                  // v = A p, rhat.v
        if (nb < 0 || tb_reduce_finish(c, nb, 1, S_TMP0)) return -1;
        hipLaunchKernelGGL(k_scalar, dim3(1), dim3(64), 0, c->s, c->scal, 2);
        hipLaunchKernelGGL(k_bicg_s, dim3(VB), dim3(VT), 0, c->s, n, r, v, sv, c->scal);
        nb = helm_apply(c, H, sv, t, true, 2);                         // t = A s, t.s, t.t
        if (nb < 0 || tb_reduce_finish(c, nb, 2, S_TS)) return -1;
        hipLaunchKernelGGL(k_scalar, dim3(1), dim3(64), 0, c->s, c->scal, 3);
        TB_PROF(c, TB_K_BICG_UPD,
                hipLaunchKernelGGL(k_bicg_xr, dim3(VB), dim3(VT), 0, c->s, n, x, r, p, sv, t, rh, c->scal, c->red));
        if (tb_reduce_finish(c, VB, 2, S_TMP1)) return -1;              // r.r, rhat.r
        hipLaunchKernelGGL(k_copy_slot, dim3(1), dim3(64), 0, c->s, c->scal, S_RHV, S_TMP2);
        TB_LAUNCH_CHECK(c);
        it++;
        if (read_scalars(c, S_TMP1, 1)) return -1;
        res = sqrt(c->hscal[S_TMP1]) / bn;
        conv = res <= rtol;
        if (!(res == res)) break;   // NaN guard
    }
    // true residual of the unscaled operator
    if (helm_apply(c, H, x, t, false, 0) < 0) return -1;
    hipLaunchKernelGGL(k_sub, dim3(VB), dim3(VT), 0, c->s, n, b, t, r, c->red);
    if (tb_reduce_finish(c, VB, 1, S_TMP1)) return -1;
    TB_CHECK(c, hipEventRecord(c->ev1, c->s));
    if (read_scalars(c, S_TMP1, 1)) return -1;
    double tres = sqrt(c->hscal[S_TMP1]) / bn;
    if (st) {
        st->iterations = it;
        st->converged = tres <= rtol;
        st->fallback = handover;
        st->vcycles = 0;
        st->res0 = res0;
        st->res = tres;
        st->ms = tb_elapsed_ms(c);
    }
    return (tres <= rtol) ? 0 : 1;
}

extern "C" int tb_helmholtz_solve(tb_ctx *c, int q, double dt, tb_solve_stats *st) {
    if (!c || q < 0 || q > 3) { if (c) c->err = "tb_helmholtz_solve: bad quantity"; return -1; }
    const HelmOp H = make_op(c, q, dt);
    TB_CHECK(c, hipEventRecord(c->ev0, c->s));
    if (c->helm_method != TB_HELM_GS) return bicgstab(c, q, H, 0, st);
    GsRun r;
    if (gs_begin(c, q, H, false, r) || gs_solve<1>(c, &r, 1, c->cfg.helm_rtol, c->cfg.helm_maxit) || gs_end(c, r)) return -1;
    if (!r.ok) return bicgstab(c, q, H, 1, st);
    gs_stats(r, tb_elapsed_ms(c), st);
    return 0;
}

// The predictor solves of a stage: u, v, w and every concentration field.
// st[q]: their stats, field 0's for the concentration (a set's time is shared
// out evenly).  Returns the worst of the solves' codes.
int tb_helmholtz_all(tb_ctx *c, double dt, tb_solve_stats *st) {
    const int sel = c->conc_sel;
    const bool set = c->helm_method == TB_HELM_GS && c->d.ntot <= HELM_SET_POINTS && tb_helm_spares(c);
    int worst = 0, first = 0;   // concentration fields from `first` on are solved one by one
    if (set) {
        GsRun run[HELM_SET];
        int n = 0;
        TB_CHECK(c, hipEventRecord(c->ev0, c->s));
        for (int q = 0; q < 3; q++, n++)
            if (gs_begin(c, q, make_op(c, q, dt), true, run[n])) return -1;
        // the IMMERSED rows of the concentration grid are those of one Pe at a time
        tb_conc_sync(c);
        bool same = true;
        for (int f = 1; f < c->nconc; f++) same &= c->cs[f].p.pe == c->cs[0].p.pe;
        if (c->nconc == 1 || same || c->nib[TB_Q_C] == 0)
            for (; first < c->nconc; first++, n++) {
                if (c->nconc > 1 && tb_conc_use(c, first)) return -1;
                if (gs_begin(c, TB_Q_C, make_op(c, TB_Q_C, dt), true, run[n])) return -1;
            }
        if (gs_solve<HELM_SET>(c, run, n, c->cfg.helm_rtol, c->cfg.helm_maxit)) return -1;
        const double ms = tb_elapsed_ms(c) / n;
        for (int a = 0; a < n; a++) {
            GsRun &r = run[a];
            if (a >= 3 && c->nconc > 1 && tb_conc_use(c, r.field)) return -1;
            tb_solve_stats s;
            if (gs_end(c, r)) return -1;
            if (r.ok) {
                gs_stats(r, ms, &s);
            } else {
                const int rc = bicgstab(c, r.q, r.H, 1, &s);
                if (rc < 0) return -1;
                if (rc > worst) worst = rc;
            }
            if (a < 3 || r.field == 0) st[r.q] = s;
        }
    }
    for (int q = 0; q < 3 && !set; q++) {
        const int rc = tb_helmholtz_solve(c, q, dt, &st[q]);
        if (rc < 0) return -1;
        if (rc > worst) worst = rc;
    }
    for (int f = first; f < c->nconc; f++) {
        if (c->nconc > 1 && tb_conc_use(c, f)) return -1;
        tb_solve_stats s;
        const int rc = tb_helmholtz_solve(c, TB_Q_C, dt, &s);
        if (rc < 0) return -1;
        if (rc > worst) worst = rc;
        if (f == 0) st[TB_Q_C] = s;
    }
    if (c->nconc > 1 && tb_conc_use(c, sel)) return -1;
    return worst;
}
