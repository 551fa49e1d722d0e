// tb_spectral.hip -- direct solve of the cell-centred Neumann -Laplacian of
// one multigrid level on its uniform box, in FP32 or FP64.
//
// The operator separates: its eigenvectors along an axis of n cells are the
// cosines cos(pi k (j + 1/2) / n) with eigenvalues (4 / h^2) sin^2(pi k / 2n).
// The solve transforms y and z to cosine modes (two dense products on the
// matrix cores), which leaves one tridiagonal system along x per (y, z) mode,
// solves those in closed form by a pair of wave-wide recurrences, and
// transforms back: five passes over the level, each reading and writing it
// once, in place after the first.  (The reference leaves this system to GMRES
// with an algebraic multigrid, Solver.c:90-265; the product form of the
// discrete Laplacian is classical: Buzbee, Golub and Nielson 1970.)
//
// At 512x256x128 in FP32 the five passes replace the five to nine
// V-cycle-preconditioned CG iterations of 0.9 ms each that one refinement
// pass of the mixed solve took.
#include <cmath>
#include <vector>

#include "tb_common.h"

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef double v4d __attribute__((ext_vector_type(4)));

template <typename T> struct V4;
template <> struct V4<float> { typedef v4f t; };
template <> struct V4<double> { typedef v4d t; };

// v_mfma_*_16x16x4: lane l holds A[l % 16][l / 16] and B[l / 16][l % 16];
// result element i of lane l is D[4 * (l / 16) + i][l % 16] in FP32 and
// D[4 * i + l / 16][l % 16] in FP64
__device__ inline v4f mfma(float a, float b, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
__device__ inline v4d mfma(double a, double b, v4d c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
__device__ inline int mfma_row(float, int lane, int i) { return 4 * (lane >> 4) + i; }
__device__ inline int mfma_row(double, int lane, int i) { return 4 * i + (lane >> 4); }

// One axis transform.  Folding the axis about its middle splits the n x n
// cosine matrix into an even and an odd half (E = ceil(n/2), O = floor(n/2)
// modes), which halves the products: the even modes see r_j + r_{n-1-j}, the
// odd ones r_j - r_{n-1-j}.  Modes are stored even ones first.
struct DctArgs {
    int n, E, O;
    int KE, KO;             // E and O rounded up to 16 (zero rows)
    long stride;            // elements between neighbours on the axis
    int ncol;               // contiguous columns per batch
    long batch;             // elements between batches
    int tiles;              // column tiles per batch
    int nblk;               // tiles * batches
};

// A block keeps NT * 16 columns of the whole axis, folded, in LDS and its four
// waves share the 16-mode tiles, each reading its matrix rows once (packed in
// the lanes' order, four steps to a 16-byte load, from L2).  The column
// index is swizzled by the row so that the four (FP64: two) rows a wave reads
// at once fall into different banks.  Bound by the matrix cores at n = 256
// (n flops per value) and by memory below n = 64; 64 columns FP32 and 32
// FP64 keep two blocks per CU up to n = 256, so one block's loads overlap
// the other's products.
template <typename T, int TN>
__device__ inline int sw(int row, int col) {
    constexpr bool f = sizeof(T) == 4;
    const int x = f && TN == 64 ? (row & 3) << 4 : f && TN == 32 ? (row & 2) << 3 : !f && TN == 32 ? (row & 1) << 4 : 0;
    return row * TN + (col ^ x);
}

template <typename T, int NT, bool INV>
__global__ void __launch_bounds__(256) k_dct(const T *in, T *out, const T *__restrict__ te,
                                             const T *__restrict__ to, DctArgs a) {
    extern __shared__ char raw[];
    T *S = reinterpret_cast<T *>(raw);
    constexpr int TN = NT * 16, RPI = 256 / TN;
    T *D = S + a.KE * TN;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int bt = blockIdx.x / a.tiles, ct = blockIdx.x - bt * a.tiles;
    const long base = bt * a.batch;
    {
        const int cc = t % TN, c = ct * TN + cc;
        const bool ok = c < a.ncol;
        const T *src = in + base + (ok ? c : 0);
#pragma unroll 4
        for (int j = t / TN; j < a.KE; j += RPI) {
            T s = (T)0, d = (T)0;
            if (INV) {
                if (ok && j < a.E) s = src[j * a.stride];
                if (ok && j < a.O) d = src[(a.E + j) * a.stride];
            } else if (ok && j < a.O) {
                const T p = src[j * a.stride], q = src[(a.n - 1 - j) * a.stride];
                s = p + q;
                d = p - q;
            } else if (ok && j < a.E) {
                s = src[j * a.stride];
            }
            S[sw<T, TN>(j, cc)] = s;
            if (j < a.KO) D[sw<T, TN>(j, cc)] = d;
        }
    }
    __syncthreads();
    typedef typename V4<T>::t vec;
    const int lr = lane >> 4, lc = lane & 15;
    // 16 rows (tile u) of one half's product with the folded columns
    auto product = [&](const T *tab, const T *B, int K, int u, vec (&acc)[NT]) {
#pragma unroll
        for (int q = 0; q < NT; q++) acc[q] = (vec){(T)0, (T)0, (T)0, (T)0};
        const vec *A = reinterpret_cast<const vec *>(tab) + (long)u * (K / 16) * 64 + lane;
        for (int kb = 0; kb < K / 16; kb++) {
            const vec av = A[kb * 64];
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const int row = kb * 16 + s * 4 + lr;
#pragma unroll
                for (int q = 0; q < NT; q++) acc[q] = mfma(av[s], B[sw<T, TN>(row, q * 16 + lc)], acc[q]);
            }
        }
    };
    const int ue = a.KE / 16, uo = a.KO / 16;
    if (!INV) {
        for (int u = wave; u < ue + uo; u += 4) {
            const bool odd = u >= ue;
            const int tile = odd ? u - ue : u;
            vec acc[NT];
            product(odd ? to : te, odd ? D : S, odd ? a.KO : a.KE, tile, acc);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int m = tile * 16 + mfma_row(T(), lane, i);
                if (m >= (odd ? a.O : a.E)) continue;
                T *dst = out + base + ((odd ? a.E : 0) + m) * a.stride;
#pragma unroll
                for (int q = 0; q < NT; q++) {
                    const int c = ct * TN + q * 16 + lc;
                    if (c < a.ncol) dst[c] = acc[q][i];
                }
            }
        }
    } else {
        for (int u = wave; u < ue; u += 4) {
            vec au[NT], av[NT];
            product(te, S, a.KE, u, au);
            if (u < uo) {
                product(to, D, a.KO, u, av);
            } else {
#pragma unroll
                for (int q = 0; q < NT; q++) av[q] = (vec){(T)0, (T)0, (T)0, (T)0};
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int m = u * 16 + mfma_row(T(), lane, i);
                if (m >= a.E) continue;
                T *lo = out + base + m * a.stride, *hi = out + base + (a.n - 1 - m) * a.stride;
#pragma unroll
                for (int q = 0; q < NT; q++) {
                    const int c = ct * TN + q * 16 + lc;
                    if (c >= a.ncol) continue;
                    lo[c] = au[q][i] + av[q][i];
                    if (m < a.O) hi[c] = au[q][i] - av[q][i];
                }
            }
        }
    }
}

// The tridiagonal systems along x, one wave per (y, z) mode, in place:
// (2 cx + mu) x_i - cx (x_{i-1} + x_{i+1}) = r_i with reflecting ends.  With
// rho the root below 1 of rho^2 - (2 + mu / cx) rho + 1 = 0 the solution on
// the evenly extended line is x_i = kappa sum_j rho^|i-j| r_j: a forward and
// a backward first-order recurrence whose end values close over the
// reflections.  Lane l runs V consecutive points, the carries cross the wave
// in six weighted shuffles; sums in FP64 in both precisions.  The (0, 0)
// mode (mu = 0) has the line's constant as its null space: its mean is
// dropped and the solution is a double prefix sum from x_0 = 0.  Reads and
// writes the level once.
struct LineArgs {
    int nx, ny, nz, px;
    long plane;
    double cx;
    const double *ly, *lz;   // eigenvalues of the stored modes
};

__device__ inline double shfl_up_d(double v, int d) { return __shfl_up(v, d, 64); }
__device__ inline double shfl_down_d(double v, int d) { return __shfl_down(v, d, 64); }

template <typename T, int V>
__global__ void __launch_bounds__(256) k_lines(T *x, LineArgs a) {
    const int lane = threadIdx.x & 63;
    const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= (long)a.ny * a.nz) return;   // whole wave
    const int j = (int)(row % a.ny), k = (int)(row / a.ny);
    T *p = x + k * a.plane + (long)j * a.px;
    const int i0 = lane * V;
    double f[V];
#pragma unroll
    for (int e = 0; e < V; e++) f[e] = i0 + e < a.nx ? (double)p[i0 + e] : 0.0;
    const double mu = a.ly[j] + a.lz[k];
    if (mu == 0.0) {
        double s = 0.0;
#pragma unroll
        for (int e = 0; e < V; e++) s += f[e];
        for (int d = 32; d > 0; d >>= 1) s += __shfl_xor(s, d, 64);
        const double mean = s / a.nx;
        // x_{i+1} - x_i = -(1/cx) sum_{j <= i} (r_j - mean)
        double g = 0.0;
#pragma unroll
        for (int e = 0; e < V; e++) {
            g += i0 + e < a.nx ? f[e] - mean : 0.0;
            f[e] = g;
        }
        double c = g;
        for (int d = 1; d < 64; d <<= 1) { const double y = shfl_up_d(c, d); if (lane >= d) c += y; }
        c = shfl_up_d(c, 1);
        if (lane == 0) c = 0.0;
        double h = 0.0;   // sum of the slopes before each point of this lane
#pragma unroll
        for (int e = 0; e < V; e++) {
            const double slope = f[e] + c;
            f[e] = h;
            h += slope;
        }
        c = h;
        for (int d = 1; d < 64; d <<= 1) { const double y = shfl_up_d(c, d); if (lane >= d) c += y; }
        c = shfl_up_d(c, 1);
        if (lane == 0) c = 0.0;
#pragma unroll
        for (int e = 0; e < V; e++)
            if (i0 + e < a.nx) p[i0 + e] = (T)(-(f[e] + c) / a.cx);
        return;
    }
    const double th = mu / a.cx, sq = sqrt(th * (1.0 + 0.25 * th));
    const double rho = 1.0 / (1.0 + 0.5 * th + sq);
    const double kappa = 1.0 / (2.0 * a.cx * sq);
    double rn = 1.0;                         // rho^nx
    {
        double b = rho;
        for (int m = a.nx; m; m >>= 1) { if (m & 1) rn *= b; b *= b; }
    }
    double w = 1.0;                          // rho^V
#pragma unroll
    for (int e = 0; e < V; e++) w *= rho;
    // local recurrences; points past the end hold 0
    double g[V];
    double s = 0.0;
#pragma unroll
    for (int e = V - 1; e >= 0; e--) { s = f[e] + rho * s; g[e] = s; }
    double cb = s;                           // backward: sum_{j >= i0} rho^(j - i0) r_j
    s = 0.0;
#pragma unroll
    for (int e = 0; e < V; e++) { const double r = f[e]; s = r + rho * s; g[e] -= r; f[e] = s; }
    double cf = s;                           // forward end of this lane
    double wd = w;
    for (int d = 1; d < 64; d <<= 1) {
        const double yf = shfl_up_d(cf, d), yb = shfl_down_d(cb, d);
        if (lane >= d) cf += wd * yf;
        if (lane + d < 64) cb += wd * yb;
        wd *= wd;
    }
    // G = sum rho^j r_j; F = sum rho^(nx-1-j) r_j, the forward value at nx - 1
    const double G = __shfl(cb, 0, 64);
    const int le = (a.nx - 1) / V;
    double pf = shfl_up_d(cf, 1), pb = shfl_down_d(cb, 1);
    if (lane == 0) pf = 0.0;
    if (lane == 63) pb = 0.0;
    double F = 0.0, wf = 1.0;
#pragma unroll
    for (int e = 0; e < V; e++) {
        wf *= rho;
        if (i0 + e == a.nx - 1) F = f[e] + wf * pf;
    }
    F = __shfl(F, le, 64);
    // values just outside the ends by reflection: f_{-1} = g_0, g_nx = f_{nx-1}
    const double g0 = (G + rn * F) / (1.0 - rn * rn);
    const double fe = F + rn * g0;
    // carries of the reflections: g0 enters lane l's forward chain with
    // rho^(l V), fe enters its backward chain with rho^(nx - (l + 1) V)
    double wl = 1.0;                         // rho^(V lane)
    {
        double b = w;
        for (int m = lane; m; m >>= 1) { if (m & 1) wl *= b; b *= b; }
    }
    const double carry_f = pf + wl * g0;
    double wr = 1.0;                         // rho^max(nx - (lane + 1) V, 0)
    {
        const int left = a.nx - (lane + 1) * V;
        double b = rho;
        for (int m = left > 0 ? left : 0; m; m >>= 1) { if (m & 1) wr *= b; b *= b; }
    }
    // the lane that holds nx - 1 takes fe at its point nx - 1, the others at
    // their last point
    const double carry_b = pb + wr * fe;
    double pw = 1.0;
#pragma unroll
    for (int e = 0; e < V; e++) { pw *= rho; f[e] += pw * carry_f; }
    const int last = a.nx - 1 - i0 < V - 1 ? a.nx - 1 - i0 : V - 1;   // this lane's last point
    pw = 1.0;
#pragma unroll
    for (int e = V - 1; e >= 0; e--) {
        if (e <= last) {
            pw *= rho;
            p[i0 + e] = (T)(kappa * (f[e] + (g[e] + pw * carry_b)));
        }
    }
}

// fragment-packed matrix: tile u, step block kb, lane l, step s hold
// M[16 u + l % 16][16 kb + 4 s + l / 16]
template <typename T, typename F>
void pack(std::vector<T> &dst, int m, int K, F value) {
    const int mt = (m + 15) / 16;
    dst.assign((size_t)mt * 16 * K, (T)0);
    for (int u = 0; u < mt; u++)
        for (int kb = 0; kb < K / 16; kb++)
            for (int l = 0; l < 64; l++)
                for (int s = 0; s < 4; s++) {
                    const int r = 16 * u + l % 16, c = 16 * kb + 4 * s + l / 16;
                    dst[(((size_t)u * (K / 16) + kb) * 64 + l) * 4 + s] = (T)value(r, c);
                }
}

inline int up16(int n) { return (n + 15) / 16 * 16; }

// LDS of one block: the folded axis for tn columns
inline long lds_bytes(int n, int tn, size_t tsize) { return (long)(up16((n + 1) / 2) + up16(n / 2)) * tn * (long)tsize; }

constexpr long LDS_TWO = 80 * 1024;    // two blocks per CU
constexpr long LDS_ONE = 156 * 1024;

// column tiles of 16 to 64 (FP64: 32) columns: the widest with two blocks per CU,
// else 16; 0: the axis does not fit
int pick_nt(int n, size_t tsize) {
    for (int nt = tsize == 4 ? 4 : 2; nt >= 1; nt >>= 1)
        if (lds_bytes(n, nt * 16, tsize) <= LDS_TWO) return nt;
    return lds_bytes(n, 16, tsize) <= LDS_ONE ? 1 : 0;
}

constexpr int X_MAX = 32 * 64;      // points of an x line in one wave's registers

template <typename T>
int build_axis(tb_ctx *c, SpecAxis &ax, int n, double h) {
    const int E = (n + 1) / 2, O = n / 2, KE = up16(E), KO = up16(O);
    auto cosine = [n](int k, int j) {
        if (k == 0) return sqrt(1.0 / n);
        // the cosine's argument reduced exactly, in quarter periods of 2n steps
        const long q = ((long)k * (2 * j + 1)) % (4L * n);
        return sqrt(2.0 / n) * cos(M_PI * (double)q / (2.0 * n));
    };
    std::vector<T> all, part;
    size_t off[4];
    for (int w = 0; w < 4; w++) {
        const bool odd = w & 1, inv = w >= 2;
        const int m = odd ? O : E, K = odd ? KO : KE;
        pack(part, m, K, [&](int r, int cc) {
            if (r >= m || cc >= m) return 0.0;
            const int mode = inv ? cc : r, j = inv ? r : cc;
            return cosine(2 * mode + (odd ? 1 : 0), j);
        });
        off[w] = all.size();
        all.insert(all.end(), part.begin(), part.end());
    }
    std::vector<double> lam(n);
    for (int p = 0; p < n; p++) {
        const int k = p < E ? 2 * p : 2 * (p - E) + 1;
        const double s = sin(M_PI * k / (2.0 * n));
        lam[p] = 4.0 / (h * h) * s * s;
    }
    ax.n = n;
    TB_CHECK(c, hipMalloc(&ax.tab, sizeof(T) * all.size()));
    TB_CHECK(c, hipMemcpy(ax.tab, all.data(), sizeof(T) * all.size(), hipMemcpyHostToDevice));
    TB_CHECK(c, hipMalloc((void **)&ax.lam, sizeof(double) * n));
    TB_CHECK(c, hipMemcpy(ax.lam, lam.data(), sizeof(double) * n, hipMemcpyHostToDevice));
    for (int w = 0; w < 4; w++) ax.off[w] = off[w];
    c->bytes += (int64_t)(sizeof(T) * all.size() + sizeof(double) * n);
    return 0;
}

template <typename T, int NT, bool INV>
void launch_nt(tb_ctx *c, const DctArgs &a, const T *in, T *out, const T *te, const T *to) {
    const int lds = (int)((a.KE + a.KO) * NT * 16 * sizeof(T));
    hipLaunchKernelGGL((k_dct<T, NT, INV>), dim3((unsigned)a.nblk), dim3(256), lds, c->s, in, out, te, to, a);
}

template <typename T, bool INV>
void dct(tb_ctx *c, const SpecAxis &ax, const T *in, T *out, long stride, int ncol, long batch, int nbatch) {
    DctArgs a;
    a.n = ax.n;
    a.E = (ax.n + 1) / 2; a.O = ax.n / 2;
    a.KE = up16(a.E); a.KO = up16(a.O);
    a.stride = stride;
    a.ncol = ncol;
    a.batch = batch;
    const int nt = pick_nt(ax.n, sizeof(T));
    a.tiles = (ncol + nt * 16 - 1) / (nt * 16);
    a.nblk = a.tiles * nbatch;
    const T *tab = (const T *)ax.tab, *te = tab + ax.off[INV ? 2 : 0], *to = tab + ax.off[INV ? 3 : 1];
    if (nt == 4) launch_nt<T, 4, INV>(c, a, in, out, te, to);
    else if (nt == 2) launch_nt<T, 2, INV>(c, a, in, out, te, to);
    else launch_nt<T, 1, INV>(c, a, in, out, te, to);
}

template <typename T, int V>
void lines_v(tb_ctx *c, T *x, const LineArgs &a) {
    const long rows = (long)a.ny * a.nz;
    hipLaunchKernelGGL((k_lines<T, V>), dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, c->s, x, a);
}

template <typename T>
int lds_attr(tb_ctx *c) {
    const void *f[6] = {(const void *)k_dct<T, 1, false>, (const void *)k_dct<T, 2, false>,
                        (const void *)k_dct<T, 4, false>, (const void *)k_dct<T, 1, true>,
                        (const void *)k_dct<T, 2, true>,  (const void *)k_dct<T, 4, true>};
    for (const void *k : f) TB_CHECK(c, hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_ONE));
    return 0;
}

}   // namespace

// whether the level's axes fit the kernels (any box up to 2048 cells along
// x and about 2400 (FP64: 1200) along y and z)
template <typename T>
bool tb_spec_usable(const Level &L) {
    return L.nx <= X_MAX && pick_nt(L.ny, sizeof(T)) > 0 && pick_nt(L.nz, sizeof(T)) > 0 &&
           (long)L.px * (L.plane / L.px) < (1L << 31) && L.ntot < (1L << 40);
}
template bool tb_spec_usable<float>(const Level &);
template bool tb_spec_usable<double>(const Level &);

// the level's matrices and eigenvalues (once)
template <typename T>
int tb_spec_build(tb_ctx *c, Level &L) {
    Spectral &s = L.spec[sizeof(T) == 8];
    if (s.z.tab) return 0;
    if (lds_attr<T>(c)) return -1;
    if (build_axis<T>(c, s.y, L.ny, L.hy) || build_axis<T>(c, s.z, L.nz, L.hz)) return -1;
    return 0;
}
template int tb_spec_build<float>(tb_ctx *, Level &);
template int tb_spec_build<double>(tb_ctx *, Level &);

void tb_spec_free(Level &L) {
    for (Spectral &s : L.spec)
        for (SpecAxis *a : {&s.y, &s.z}) {
            hipFree(a->tab);
            hipFree(a->lam);
            *a = SpecAxis();
        }
}

// out = A^+ in on the level's cells (in its layout; entries outside the cells
// are neither needed nor kept), up to a constant; in and out distinct
template <typename T>
int tb_spec_solve(tb_ctx *c, const Level &L, const T *in, T *out) {
    const Spectral &s = L.spec[sizeof(T) == 8];
    const int zcol = L.px * (L.ny - 1) + L.nx;   // columns of a plane up to its last cell
    dct<T, false>(c, s.y, in, out, L.px, L.nx, L.plane, L.nz);
    dct<T, false>(c, s.z, out, out, L.plane, zcol, 0, 1);
    LineArgs a;
    a.nx = L.nx; a.ny = L.ny; a.nz = L.nz; a.px = L.px; a.plane = L.plane;
    a.cx = 1.0 / (L.hx * L.hx);
    a.ly = s.y.lam; a.lz = s.z.lam;
    if (L.nx <= 64) lines_v<T, 1>(c, out, a);
    else if (L.nx <= 128) lines_v<T, 2>(c, out, a);
    else if (L.nx <= 256) lines_v<T, 4>(c, out, a);
    else if (L.nx <= 512) lines_v<T, 8>(c, out, a);
    else if (L.nx <= 1024) lines_v<T, 16>(c, out, a);
    else lines_v<T, 32>(c, out, a);
    dct<T, true>(c, s.z, out, out, L.plane, zcol, 0, 1);
    dct<T, true>(c, s.y, out, out, L.px, L.nx, L.plane, L.nz);
    TB_LAUNCH_CHECK(c);
    return 0;
}
template int tb_spec_solve<float>(tb_ctx *, const Level &, const float *, float *);
template int tb_spec_solve<double>(tb_ctx *, const Level &, const double *, double *);
