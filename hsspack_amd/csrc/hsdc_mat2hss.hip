// Dense matrix -> HSS form by truncated SVDs on gfx950: the construction half of
// HSSPACK's DHSSMM / DHSSMML (DHSSMM.f90:1-125, DHSSMML.f90:2-122; mat2hssvd,
// ConstructHssd.f90:371-696), done depth by depth.  The compressed matrix C holds, for
// the active nodes in left-to-right order, C(a, b) = U_a^T A(a, b) W_b (a raw leaf's
// basis is the identity).  For every node of one depth, all in one launch:
//
//   k_m2h_gather   its block row (its rows against the other active columns) transposed
//                  and its block column, as tall matrices (context x own)
//   k_m2h_qr       contexts of many rows reduced first by a tree of QRs in LDS
//   k_m2h_svd      one workgroup per (node, side): Householder QR of the tall matrix and
//                  one-sided Jacobi, on the transposed triangle of a second QR or, for a
//                  sketch, on R's columns with the rotations accumulated (the right
//                  singular vectors); for a matrix wider than tall the columns of
//                  its transpose are orthogonalised directly; the singular values
//                  descending, the rank = their count above tol (mat2hssvd's
//                  count(svs > tol)), the basis vectors in that order
//   k_m2h_rows,    C' = blockdiag(U)^T C blockdiag(W) over the new active list, one output
//   k_m2h_cols     element per thread
//   k_m2h_copy     generators: U (m x r), V = W^T (r x m), each sibling pair's B from C'
//
// With randomized range finding (mat2hssvdr), k_m2h_sketch forms Omega T for each side
// with a long context before k_m2h_svd, which then decomposes the sketch.
//
// The generators land in the layout the HSS multiply reads (U, V^T, B, D per node, the
// post-ordered tree of npart), so DHSSMM and DHSSMML run the same batched multiply as
// the eigenvector matrices.
#include <float.h>
#include <math.h>
#include "hsdc_internal.h"
#include "hsdc_m2h.h"

#define MWG 256

namespace {

__device__ __forceinline__ int m2h_rr(int slot, int r, int P)
{
    if (slot == 0) return 0;
    return 1 + (slot - 1 + (P - 1) - (r % (P - 1))) % (P - 1);
}

}  // namespace

// ---------------------------------------------------------------------------
// Gather the tall matrices: side 0: T(o, t) = C(rs + t, col_o), col_o the o-th column
// outside [cs, cs + cn); side 1: T(o, t) = C(row_o, cs + t), row_o outside [rs, rs + rn).
// Grid: (chunks, jobs); one thread per element.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(MWG) void k_m2h_gather(const M2hJob *jobs, const double *C, long ldc, double *S)
{
    const M2hJob J = jobs[blockIdx.y];
    const int side = blockIdx.y & 1;
    const long tot = (long)J.w * J.m;
    double *T = S + J.toff;
    for (long e = (long)blockIdx.x * MWG + threadIdx.x; e < tot; e += (long)gridDim.x * MWG) {
        const int o = (int)(e % J.w), t = (int)(e / J.w);
        if (side == 0) {
            const int col = o < J.cs ? o : o + J.cn;
            T[e] = C[(J.rs + t) + (long)col * ldc];
        } else {
            const int row = o < J.rs ? o : o + J.rn;
            T[e] = C[row + (long)(J.cs + t) * ldc];
        }
    }
}

// ---------------------------------------------------------------------------
// One workgroup per job.  w >= m: Householder QR of T in place (v = (1, x(1:)), tau =
// (beta - alpha) / beta, beta = -sign(alpha) |x|), R's upper triangle copied to the R
// area, then one-sided Jacobi on its m columns with the rotations accumulated in V
// (identity at the start); the basis = V's columns by descending column norm of the
// rotated R.  w < m: the m x w transpose of T is copied to the R area and its w columns
// orthogonalised; the basis = the normalised columns by descending norm (the rest zero).
// A pair rotates when |c_a . c_b| > L eps |c_a| |c_b|, L the column length; 60 sweeps at
// most (else *err is set).  rank[job] = the count of singular values above tol.
//
// The bound is the latency of the sweeps: m - 1 rounds of m / 2 pairs, about ten sweeps,
// each pair three dot products and a chain of square roots and divides.  Sixteen
// wavefronts take a pair each, and R and V stay in LDS as far as lds_cap doubles hold
// them (R and V up to m = 99, R alone up to m = 140, else global memory).  With four
// wavefronts and R and V in global memory a level of the n = 2000, leaf 64 matrix took
// 26 ms.
// ---------------------------------------------------------------------------
typedef __attribute__((address_space(3))) double m2h_ldbl;
typedef __attribute__((address_space(1))) double m2h_gdbl;

// Jacobi on the P columns of R (length m, ld m), with V when qr; then the singular values
// (column norms) to sv, their descending order (ties by index) to ord, the basis to B.
// Returns false when the sweeps did not converge or the matrix's norm is no finite number
// (B, sv and ord may then be unset).
template <class RP, class VP>
__device__ __forceinline__ bool m2h_jacobi(RP R, VP V, bool qr, int m, int P, double *sv, int *ord, double *B,
                                           int *s_rot, double *s_part)
{
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, NW = M2H_SVD_WG / 64;
    const int L = m, PP = P + (P & 1);
    bool conv = P < 2;
    // Columns parallel to the last bit (a block of exact rank one) stay parallel: every
    // sweep only shrinks the smaller by about eps, and once the squares are denormal the
    // angles are noise and the sweeps never end.  A column below 2^-300 of the matrix's norm
    // is left alone.
    double part = 0.0;
    for (long e = tid; e < (long)m * P; e += M2H_SVD_WG) part += R[e] * R[e];
    part = team_bfly(part, 64);
    if (lane == 0) s_part[wv] = part;
    __syncthreads();
    double lim = 0.0;
    for (int q = 0; q < NW; q++) lim += s_part[q];
    // A NaN, an infinity or an overflow among the squares: no angles and no order of the
    // singular values; the caller multiplies densely.  Rotations keep the sum, so a norm
    // below is a number whenever this test passes.
    if (!(lim <= DBL_MAX)) return false;
    lim *= 0x1p-600;
    for (int sweep = 0; sweep < 60 && !conv; sweep++) {
        if (tid == 0) *s_rot = 0;
        __syncthreads();
        bool rot = false;
        for (int r = 0; r < PP - 1; r++) {
            // two pairs per wavefront at a time: their sums and rotations overlap
            for (int pr = wv; pr < PP / 2; pr += 2 * NW) {
                int pa[2], pb[2];
                bool ok[2];
                double al[2] = {0.0, 0.0}, be[2] = {0.0, 0.0}, ga[2] = {0.0, 0.0}, cc[2], ss[2];
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const int q = pr + u * NW;
                    const int x = m2h_rr(q, r, PP), y = m2h_rr(PP - 1 - q, r, PP);
                    pa[u] = x < y ? x : y;
                    pb[u] = x < y ? y : x;
                    ok[u] = q < PP / 2 && pb[u] < P;  // uniform over the wavefront
                }
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    if (!ok[u]) continue;
                    const RP ca = R + (long)pa[u] * m, cb = R + (long)pb[u] * m;
                    for (int k = lane; k < L; k += 64) {
                        const double x = ca[k], y = cb[k];
                        al[u] += x * x; be[u] += y * y; ga[u] += x * y;
                    }
                }
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    al[u] = team_bfly(al[u], 64); be[u] = team_bfly(be[u], 64); ga[u] = team_bfly(ga[u], 64);
                }
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    if (ga[u] == 0.0 || fmin(al[u], be[u]) <= lim ||
                        !(fabs(ga[u]) > L * HSDC_EPS * sqrt(al[u] * be[u])))
                        ok[u] = false;
                    const double ze = (be[u] - al[u]) / (2.0 * ga[u]);
                    const double t = (ze >= 0.0 ? 1.0 : -1.0) / (fabs(ze) + sqrt(1.0 + ze * ze));
                    cc[u] = 1.0 / sqrt(1.0 + t * t);
                    ss[u] = cc[u] * t;
                }
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    if (!ok[u]) continue;
                    const RP ca = R + (long)pa[u] * m, cb = R + (long)pb[u] * m;
                    for (int k = lane; k < L; k += 64) {
                        const double x = ca[k], y = cb[k];
                        ca[k] = cc[u] * x - ss[u] * y;
                        cb[k] = ss[u] * x + cc[u] * y;
                    }
                    if (qr) {
                        const VP va = V + (long)pa[u] * m, vb = V + (long)pb[u] * m;
                        for (int k = lane; k < m; k += 64) {
                            const double x = va[k], y = vb[k];
                            va[k] = cc[u] * x - ss[u] * y;
                            vb[k] = ss[u] * x + cc[u] * y;
                        }
                    }
                    rot = true;
                }
            }
            __syncthreads();
        }
        if (rot && lane == 0) *s_rot = 1;
        __syncthreads();
        conv = (*s_rot == 0);
        __syncthreads();
    }
    for (int j = wv; j < P; j += NW) {
        double q = 0.0;
        for (int k = lane; k < L; k += 64) q += R[k + (long)j * m] * R[k + (long)j * m];
        q = sqrt(team_bfly(q, 64));
        if (lane == 0) sv[j] = q;
    }
    __syncthreads();
    // positions by counting, ties by index: a permutation because the keys are totally ordered
    // (a NaN would be the smallest)
    auto key = [&](int j) { const double q = sv[j]; return q >= 0.0 ? q : -1.0; };
    for (int j = tid; j < P; j += M2H_SVD_WG) {
        const double x = key(j);
        int rk = 0;
        for (int i = 0; i < P; i++) {
            const double y = key(i);
            rk += (y > x || (y == x && i < j)) ? 1 : 0;
        }
        ord[rk] = j;
    }
    __syncthreads();
    for (long e = tid; e < (long)m * m; e += M2H_SVD_WG) {
        const int i = (int)(e % m), j = (int)(e / m);
        double v = 0.0;
        if (j < P) {
            const int s0 = ord[j];
            if (qr) v = V[i + (long)s0 * m];
            else {
                const double nrm = sv[s0];
                v = nrm > 0.0 ? R[i + (long)s0 * m] / nrm : 0.0;
            }
        }
        B[e] = v;
    }
    return conv;
}

// Householder QR of T (w x m in LDS, ld w, m <= w <= M2H_QR_ROWS, m <= M2H_QM) in place: R's
// part above the diagonal in T, its diagonal in rdiag.  Every wavefront forms the reflector
// of a column by itself (its rows in registers) and applies it to its share of the columns,
// so a column takes one barrier.  The reflectors I - rtau v v^T stay as v(1:) = rsc times T's part below
// the diagonal.  A barrier precedes the return.
__device__ __forceinline__ void m2h_qr_lds(m2h_ldbl *T, int w, int m, double *rdiag, double *rsc, double *rtau)
{
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, NW = M2H_SVD_WG / 64;
    for (int k = 0; k < m; k++) {
        const m2h_ldbl *x = T + k + (long)k * w;
        const int len = w - k;
        double v[8], part = 0.0;
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const int i = 1 + lane + 64 * q;
            v[q] = i < len ? x[i] : 0.0;
            part += v[q] * v[q];
        }
        const double xn = sqrt(team_bfly(part, 64)), alpha = x[0];
        double diag = alpha, rs = 0.0, rt = 0.0;
        if (xn != 0.0) {  // else H = I
            const double beta = -copysign(hypot(alpha, xn), alpha);
            const double tau = (beta - alpha) / beta, scal = 1.0 / (alpha - beta);
#pragma unroll
            for (int q = 0; q < 8; q++) v[q] *= scal;
            for (int j = k + 1 + wv; j < m; j += NW) {
                m2h_ldbl *c = T + k + (long)j * w;
                double cv[8], d = 0.0;
                const double c0 = c[0];
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    const int i = 1 + lane + 64 * q;
                    cv[q] = i < len ? c[i] : 0.0;
                    d += v[q] * cv[q];
                }
                d = (c0 + team_bfly(d, 64)) * tau;
                if (lane == 0) c[0] = c0 - d;
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    const int i = 1 + lane + 64 * q;
                    if (i < len) c[i] = cv[q] - d * v[q];
                }
            }
            diag = beta;
            rs = scal;
            rt = tau;
        }
        if (threadIdx.x == 0) { rdiag[k] = diag; rsc[k] = rs; rtau[k] = rt; }
        __syncthreads();
    }
}

// V := Q of the QR above for a square matrix (w = m <= 128): the reflectors applied to the
// identity, a column per wavefront in registers, four columns at a time.
__device__ __forceinline__ void m2h_q_form(const m2h_ldbl *T, m2h_ldbl *V, int m, const double *rsc, const double *rtau)
{
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, NW = M2H_SVD_WG / 64;
    for (int j0 = wv; j0 < m; j0 += 4 * NW) {
        double c[4][2];
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int q = 0; q < 2; q++) c[t][q] = lane + 64 * q == j0 + t * NW ? 1.0 : 0.0;
        for (int k = m - 1; k >= 0; k--) {
            const double sc = rsc[k], tau = rtau[k];
            double v[2], d[4];
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const int i = lane + 64 * q;
                v[q] = i == k ? 1.0 : (i > k && i < m) ? T[i + k * m] * sc : 0.0;
            }
#pragma unroll
            for (int t = 0; t < 4; t++) d[t] = team_bfly(v[0] * c[t][0] + v[1] * c[t][1], 64);
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int q = 0; q < 2; q++) c[t][q] -= d[t] * tau * v[q];
        }
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const int i = lane + 64 * q, j = j0 + t * NW;
                if (i < m && j < m) V[i + j * m] = c[t][q];
            }
    }
}

// One chunk of rows of a tall matrix (rows x m at src, ld lds) reduced to its R (m x m at
// dst, ld ldd): the tree reduction that brings a context of thousands of rows down to what
// k_m2h_svd holds in LDS.  One workgroup walking the whole matrix in global memory took
// about 7 ms for 1936 x 64, with most CUs idle.
__global__ __launch_bounds__(M2H_SVD_WG) void k_m2h_qr(const M2hChunk *ch, double *S)
{
    extern __shared__ double m2h_dyn[];
    __shared__ double rdiag[M2H_QM], rsc[M2H_QM], rtau[M2H_QM];
    const M2hChunk C = ch[blockIdx.x];
    m2h_ldbl *T = (m2h_ldbl *)m2h_dyn;
    const double *src = S + C.src;
    double *dst = S + C.dst;
    for (int e = threadIdx.x; e < C.rows * C.m; e += M2H_SVD_WG)
        T[e] = src[(e % C.rows) + (long)(e / C.rows) * C.lds];
    __syncthreads();
    m2h_qr_lds(T, C.rows, C.m, rdiag, rsc, rtau);
    for (int e = threadIdx.x; e < C.m * C.m; e += M2H_SVD_WG) {
        const int i = e % C.m, j = e / C.m;
        dst[i + (long)j * C.ldd] = i < j ? T[i + (long)j * C.rows] : i == j ? rdiag[j] : 0.0;
    }
}

__global__ __launch_bounds__(M2H_SVD_WG) void k_m2h_svd(const M2hJob *jobs, double *S, double *Bs, double tol, int *rank,
                                                        int *err, int lds_cap)
{
    extern __shared__ double m2h_dyn[];  // lds_cap doubles
    __shared__ double red[M2H_SVD_WG / 64];
    __shared__ int s_rot, s_cnt;
    const M2hJob J = jobs[blockIdx.x];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, NW = M2H_SVD_WG / 64;
    const int w = J.w, m = J.m;
    double *T = S + J.toff, *Rg = T + (long)w * m, *Vg = Rg + (long)m * m;
    double *B = Bs + J.boff, *sv = B + (long)m * m;
    int *ord = (int *)(sv + m);  // P ints after the singular values
    const bool qr = w >= m;
    const int P = qr ? m : w;  // columns of length m to orthogonalise
    const long rsz = (long)m * P;
    const bool rl = rsz <= lds_cap, vl = rl && qr && rsz + (long)m * m <= lds_cap;
    m2h_ldbl *Rl = (m2h_ldbl *)m2h_dyn, *Vl = Rl + rsz;
    if (qr && vl && w <= M2H_QR_ROWS && (long)w * m <= lds_cap) {
        // The matrix itself in LDS, then R over it.  With lq the sweeps run on L = R3^T of a
        // second QR, R^T = Q3 R3, with the rotations accumulated on Q3: T = Q L Q3^T, and the
        // rows of R3 are graded, which takes 9 sweeps where R takes 21 (64 columns of the
        // Cauchy test matrix).  Leaving pairs of columns below tol alone would save rotations,
        // but near a spectrum that is dense around tol it never converges.
        // Not for a sketch: its largest singular value is so much above the block's that
        // eps sigma_1 is a sizeable part of tol, and another QR's rounding moves the rank.
        __shared__ double rdiag[M2H_QM], rsc[M2H_QM], rtau[M2H_QM];
        constexpr int NE = M2H_QM * M2H_QM / M2H_SVD_WG + 1;  // elements of an m x m matrix per thread
        double r[NE];
        for (int e = tid; e < w * m; e += M2H_SVD_WG) Rl[e] = T[e];
        __syncthreads();
        m2h_qr_lds(Rl, w, m, rdiag, rsc, rtau);
        // the triangle a QR leaves (ld ldr) or its transpose to the front of the LDS
        auto triangle = [&](int ldr, bool tr) {
#pragma unroll
            for (int q = 0; q < NE; q++) {
                const int e = tid + q * M2H_SVD_WG, i = tr ? e / m : e % m, j = tr ? e % m : e / m;
                r[q] = e < m * m ? (i < j ? Rl[i + j * ldr] : i == j ? rdiag[j] : 0.0) : 0.0;
            }
            __syncthreads();
#pragma unroll
            for (int q = 0; q < NE; q++) {
                const int e = tid + q * M2H_SVD_WG;
                if (e < m * m) Rl[e] = r[q];
            }
            __syncthreads();
        };
        triangle(w, J.lq != 0);
        if (J.lq) {
            m2h_qr_lds(Rl, m, m, rdiag, rsc, rtau);
            m2h_q_form(Rl, Vl, m, rsc, rtau);
            __syncthreads();
            triangle(m, true);
        } else {
            for (int e = tid; e < m * m; e += M2H_SVD_WG) Vl[e] = (e % m == e / m) ? 1.0 : 0.0;
        }
    } else if (qr) {
        for (int k = 0; k < m; k++) {
            double *x = T + k + (long)k * w;
            const int len = w - k;
            double part = 0.0;
            for (int i = 1 + tid; i < len; i += M2H_SVD_WG) part += x[i] * x[i];
            part = team_bfly(part, 64);
            if (lane == 0) red[wv] = part;
            __syncthreads();
            double xn = 0.0;
            for (int q = 0; q < NW; q++) xn += red[q];
            xn = sqrt(xn);
            const double alpha = x[0];
            __syncthreads();
            if (xn == 0.0) continue;  // uniform: H = I
            const double beta = -copysign(hypot(alpha, xn), alpha);
            const double tau = (beta - alpha) / beta, scal = 1.0 / (alpha - beta);
            for (int i = 1 + tid; i < len; i += M2H_SVD_WG) x[i] *= scal;
            __syncthreads();
            for (int j = k + 1 + wv; j < m; j += NW) {
                double *c = T + k + (long)j * w;
                double d = 0.0;
                for (int i = 1 + lane; i < len; i += 64) d += x[i] * c[i];
                d = team_bfly(d, 64);
                d = (c[0] + d) * tau;
                if (lane == 0) c[0] -= d;
                for (int i = 1 + lane; i < len; i += 64) c[i] -= d * x[i];
            }
            __syncthreads();
            if (tid == 0) x[0] = beta;
            __syncthreads();
        }
        for (long e = tid; e < (long)m * m; e += M2H_SVD_WG) {
            const int i = (int)(e % m), j = (int)(e / m);
            const double r = (i <= j) ? T[i + (long)j * w] : 0.0, v = (i == j) ? 1.0 : 0.0;
            if (rl) Rl[e] = r; else Rg[e] = r;
            if (vl) Vl[e] = v; else Vg[e] = v;
        }
    } else {
        for (long e = tid; e < rsz; e += M2H_SVD_WG) {
            const int i = (int)(e % m), j = (int)(e / m);  // R area as m x w: column j = row j of T
            const double r = T[j + (long)i * w];
            if (rl) Rl[e] = r; else Rg[e] = r;
        }
    }
    if (tid == 0) s_cnt = 0;
    __syncthreads();
    bool conv;
    m2h_gdbl *Rq = (m2h_gdbl *)Rg, *Vq = (m2h_gdbl *)Vg;
    if (vl) conv = m2h_jacobi(Rl, Vl, qr, m, P, sv, ord, B, &s_rot, red);
    else if (rl) conv = m2h_jacobi(Rl, Vq, qr, m, P, sv, ord, B, &s_rot, red);
    else conv = m2h_jacobi(Rq, Vq, qr, m, P, sv, ord, B, &s_rot, red);
    if (!conv) {  // uniform; the host then reads neither the rank nor the basis
        if (tid == 0) { atomicOr(err, 1); rank[blockIdx.x] = 0; }
        return;
    }
    for (int j = tid; j < P; j += M2H_SVD_WG)
        if (sv[j] > tol) atomicAdd(&s_cnt, 1);
    __syncthreads();
    if (tid == 0) rank[blockIdx.x] = s_cnt;
}

// ---------------------------------------------------------------------------
// Randomized range finding (mat2hssvdr, ConstructHssd.f90:8-368): a side whose context
// is longer than 50 and than m + 10 takes its basis from the sketch Omega T (pp x m,
// pp = m + 10) instead of T.  The reference draws one flat array of uniform [0, 1)
// numbers and reads it as a pp x w matrix (leading dimension pp) for a block column and
// as a w x pp matrix (leading dimension w) for a block row (:104, :129, ...); entry i of
// the flat array here is m2h_omega(seed, i), the splitmix64 stream of the seed, so the
// oracle draws the same numbers.  sk[job] is the sketch job (w = pp, toff at its
// scratch) or the job itself.  Grid: (chunks, jobs); one thread per element of S.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double m2h_omega(unsigned long long seed, unsigned long long i)
{
    unsigned long long z = seed + 0x9E3779B97F4A7C15ull * (i + 1);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (double)(z >> 11) * 0x1p-53;
}

__global__ __launch_bounds__(MWG) void k_m2h_sketch(const M2hJob *jobs, const M2hJob *sk, const double *S0, double *S,
                                                    unsigned long long seed)
{
    const M2hJob J = jobs[blockIdx.y], K = sk[blockIdx.y];
    if (K.lq) return;  // no sketch for this side (a tree of QRs may have changed its width)
    const int side = blockIdx.y & 1, pp = K.w, w = J.w;
    const double *T = S0 + J.toff;
    double *Y = S + K.toff;
    const long tot = (long)pp * J.m;
    for (long e = (long)blockIdx.x * MWG + threadIdx.x; e < tot; e += (long)gridDim.x * MWG) {
        const int r = (int)(e % pp), t = (int)(e / pp);
        const double *tc = T + (long)t * w;
        double acc = 0.0;
        for (int o = 0; o < w; o++) {
            const unsigned long long idx = side ? (unsigned long long)r + (unsigned long long)o * pp
                                                : (unsigned long long)o + (unsigned long long)r * w;
            acc += m2h_omega(seed, idx) * tc[o];
        }
        Y[e] = acc;
    }
}

// New rows of C: for each new row block a, U_q^T C(rows of q, :) when it comes from a
// job pair q (src >= 0), the old rows otherwise.  out is nnr x nc (ld nnr).
__global__ __launch_bounds__(MWG) void k_m2h_rows(const M2hBlk *blk, int nb, const M2hJob *jobs, const double *Bs,
                                                  const double *C, long ldc, int nc, double *out, long ldo)
{
    const long tot = ldo * (long)nc;
    for (long e = (long)blockIdx.x * MWG + threadIdx.x; e < tot; e += (long)gridDim.x * MWG) {
        const int r = (int)(e % ldo), c = (int)(e / ldo);
        int lo = 0, hi = nb - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (blk[mid].start <= r) lo = mid; else hi = mid - 1;
        }
        const M2hBlk b = blk[lo];
        const int i = r - b.start;
        double v;
        if (b.src >= 0) {
            const M2hJob J = jobs[2 * b.src];
            const double *U = Bs + J.boff;  // m x m, column i
            v = 0.0;
            for (int t = 0; t < J.m; t++) v += U[t + (long)i * J.m] * C[(b.ostart + t) + (long)c * ldc];
        } else {
            v = C[(b.ostart + i) + (long)c * ldc];
        }
        out[r + (long)c * ldo] = v;
    }
}

// New columns: C'(:, new block b) = Tr(:, old columns of q) W_q, or a copy.
__global__ __launch_bounds__(MWG) void k_m2h_cols(const M2hBlk *blk, int nb, const M2hJob *jobs, const double *Bs,
                                                  const double *Tr, long ldt, int nnc, double *out)
{
    const long tot = ldt * (long)nnc;
    for (long e = (long)blockIdx.x * MWG + threadIdx.x; e < tot; e += (long)gridDim.x * MWG) {
        const int r = (int)(e % ldt), c = (int)(e / ldt);
        int lo = 0, hi = nb - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (blk[mid].start <= c) lo = mid; else hi = mid - 1;
        }
        const M2hBlk b = blk[lo];
        const int j = c - b.start;
        double v;
        if (b.src >= 0) {
            const M2hJob J = jobs[2 * b.src + 1];
            const double *W = Bs + J.boff;  // m x m, column j
            v = 0.0;
            for (int t = 0; t < J.m; t++) v += Tr[r + (long)(b.ostart + t) * ldt] * W[t + (long)j * J.m];
        } else {
            v = Tr[r + (long)(b.ostart + j) * ldt];
        }
        out[r + (long)c * ldt] = v;
    }
}

// Copies of one level's generators into the arena (M2hCopy).
__global__ __launch_bounds__(MWG) void k_m2h_copy(const M2hCopy *cp, const M2hJob *jobs, const double *Bs,
                                                  const double *Cn, long ldcn, const double *A, long lda,
                                                  double *arena, double *dd)
{
    const M2hCopy P = cp[blockIdx.y];
    const long tot = (long)P.rows * P.cols;
    double *dst = (P.kind == 3 ? dd : arena) + P.dst;
    for (long e = (long)blockIdx.x * MWG + threadIdx.x; e < tot; e += (long)gridDim.x * MWG) {
        const int i = (int)(e % P.rows), j = (int)(e / P.rows);
        double v;
        if (P.kind == 0) {
            const M2hJob J = jobs[P.job];
            v = Bs[J.boff + i + (long)j * J.m];
        } else if (P.kind == 1) {
            const M2hJob J = jobs[P.job];
            v = Bs[J.boff + j + (long)i * J.m];
        } else if (P.kind == 2) {
            v = Cn[(P.r0 + i) + (long)(P.c0 + j) * ldcn];
        } else {
            v = A[(P.r0 + i) + (long)(P.c0 + j) * lda];
        }
        dst[e] = v;
    }
}
