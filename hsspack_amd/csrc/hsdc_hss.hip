// HSS form of the eigenvector matrix of a rank-one merge and its product with the
// old eigenvectors, for gfx950.
//
//   construction  Cauchy2hssEig_omp / ComprcauchyEig / rrluCauchyEigrow,col
//                 (CauchyHssEig.f90:7-467, 1945-2440): one workgroup per HSS node
//                 runs the structured rank-revealing LU on the Cauchy generators;
//                 every element of the Schur complement it touches is formed from
//                 the generators with the accurate differences of
//                 computfd / computdd (CauchyHssEig.f90:470-568), so nothing of the
//                 K x K matrix is ever stored.  Statement order follows the
//                 reference, which keeps pivots, ranks and generators identical to
//                 the CPU oracle's restatement.
//   multiply      fastHssmmL_omp (ConstructHssd.f90:1394-1630): X := X * H as
//                 batched FP64 MFMA GEMMs, one launch per tree level, over all
//                 nodes of all HSS merges of the DC level and all row tiles of X.
#include <float.h>
#include "hsdc_internal.h"
#include "hsdc_hss.h"

#define WG 256
#define A1(a, i) (a)[(i) - 1]
#define HSS_RB 2  // outside columns a thread takes at a time in the RRLU passes

// Pointers typed by address space: global memory (1) and LDS (3).  Loads through an
// untyped pointer compile to FLAT instructions, which the compiler must order against
// every LDS access and every store; typed loads and stores let it issue the loads of
// many columns before their results are needed.
typedef const __attribute__((address_space(1))) double gdbl;
typedef __attribute__((address_space(1))) double gdblw;
typedef __attribute__((address_space(1))) int gint;
typedef const __attribute__((address_space(1))) int gcint;
typedef __attribute__((address_space(3))) double ldbl;

// ---------------------------------------------------------------------------
// accurate differences: f_{PL(j)} - lambda_{PU(k)} and lambda_{PU(j)} - lambda_{PU(k)}
// ---------------------------------------------------------------------------
__device__ __forceinline__ double fd(const HssMerge &H, int pd, int pw)
{
    gdbl *FF = (gdbl *)H.FF;
    if (pd <= pw) return (A1(FF, pd) - A1(FF, pw)) - A1((gdbl *)H.DIFL, pw);
    return (A1(FF, pd) - A1(FF, pw + 1)) - A1((gdbl *)H.DIFR, pw);
}
__device__ __forceinline__ double dd(const HssMerge &H, int pj, int pk)
{
    gdbl *FF = (gdbl *)H.FF;
    if (pj < pk) return ((A1(FF, pj + 1) - A1(FF, pk)) + A1((gdbl *)H.DIFR, pj)) - A1((gdbl *)H.DIFL, pk);
    return ((A1(FF, pj) - A1(FF, pk + 1)) + A1((gdbl *)H.DIFL, pj)) - A1((gdbl *)H.DIFR, pk);
}

// The same differences from values gathered once per root: a pass over many columns
// loads, for each column's root p, FF(p), FF(p + 1), DIFL(p), DIFR(p) (and D0(p) for the
// squared form) together, then forms every difference it needs from registers.  The
// operations and their order are those of fd / dd above, so the results are identical.
struct RootG { double f0, f1, dl, dr, s; };
template <bool SQ>
__device__ __forceinline__ RootG root_load(const HssMerge &H, int p)
{
    RootG r;
    r.f0 = A1((gdbl *)H.FF, p);
    r.f1 = A1((gdbl *)H.FF, p < H.K ? p + 1 : p);  // FF(p + 1) is read only for p < K
    r.dl = A1((gdbl *)H.DIFL, p);
    r.dr = A1((gdbl *)H.DIFR, p);
    r.s = SQ ? A1((gdbl *)H.D0, p) : 0.0;
    return r;
}
// fdq(pd, pw) with ffd = FF(pd) and w = root_load(pw)
template <bool SQ>
__device__ __forceinline__ double fd_r(double ffd, int pd, int pw, const RootG &w)
{
    const double r = (pd <= pw) ? (ffd - w.f0) - w.dl : (ffd - w.f1) - w.dr;
    return SQ ? r * (ffd + w.s) : r;
}
// Whether |z / den| can exceed the running maximum mv of a "first largest" search: the
// hardware reciprocal gives |z| / |den| to far better than 2^-10 relative, so an entry
// estimated below mv (1 - 2^-10) is below mv exactly and cannot replace it; every other
// entry (and any zero, infinite or NaN operand) takes the exact division.  The searches
// therefore choose the same entries as with a division for every element.
__device__ __forceinline__ bool may_exceed(double z, double den, double mv)
{
    const double az = fabs(z);
    const double ap = az * __builtin_amdgcn_rcp(fabs(den));
    return !(ap < mv * (1.0 - 0x1p-10)) || (ap == 0.0 && az != 0.0);
}
// ddq(pj, pk) with j = root_load(pj), k = root_load(pk)
template <bool SQ>
__device__ __forceinline__ double dd_r(int pj, const RootG &j, int pk, const RootG &k)
{
    const double r = (pj < pk) ? ((j.f1 - k.f0) + j.dr) - k.dl : ((j.f0 - k.f1) + j.dl) - k.dr;
    return SQ ? r * (j.s + k.s) : r;
}
// The SVD's vector matrices u_i v_j / (f_i^2 - sigma_j^2) are Cauchy-like in the
// squared variables: with SQ every displacement is the accurate difference times the
// sum (D0 holds the roots sigma): pole-root, root-root and pole-pole.
template <bool SQ>
__device__ __forceinline__ double fdq(const HssMerge &H, int pd, int pw)
{
    const double r = fd(H, pd, pw);
    return SQ ? r * (A1((gdbl *)H.FF, pd) + A1((gdbl *)H.D0, pw)) : r;
}
template <bool SQ>
__device__ __forceinline__ double ddq(const HssMerge &H, int pj, int pk)
{
    const double r = dd(H, pj, pk);
    return SQ ? r * (A1((gdbl *)H.D0, pj) + A1((gdbl *)H.D0, pk)) : r;
}
template <bool SQ>
__device__ __forceinline__ double ppq(double a, double b)
{
    return SQ ? (a - b) * (a + b) : a - b;
}

// block-wide (max |value|, first index); idx <= 0 means "no entry"
struct VI { double v; int i; };
__device__ __forceinline__ VI vi_better(VI a, VI b)
{
    if (b.i <= 0) return a;
    if (a.i <= 0) return b;
    if (b.v > a.v || (b.v == a.v && b.i < a.i)) return b;
    return a;
}
template <int O>
__device__ __forceinline__ VI vi_step(VI x)
{
    VI y;
    y.v = xlane<O>(x.v);
    y.i = xlane32<O>(x.i);
    return vi_better(x, y);
}
// v of the lane CTRL names, or v itself where that lane is outside the row
template <int CTRL>
__device__ __forceinline__ double dpp_max(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = (int)(unsigned)b, hi = (int)(b >> 32);
    const int l2 = __builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xF, 0xF, false);
    const int h2 = __builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xF, 0xF, false);
    return fmax(v, __longlong_as_double(((long long)h2 << 32) | (unsigned)l2));
}
__device__ __forceinline__ double lane_value(double v, int l)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(unsigned)b, l);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// The (value, smallest index) maximum over the wavefront's first NL lanes (4 to 64), in
// every lane, for values >= 0: the values go through a prefix of DPP moves (no LDS
// traffic), the index is read from the lane a ballot finds.  A butterfly of (value,
// index) pairs, three of whose six steps cross lanes through LDS, took about 1000 cycles
// for two reductions; this takes about 300.
template <int NL>
__device__ __forceinline__ VI wave_argmax(VI x)
{
    const double v = x.i > 0 ? x.v : -1.0;
    double m = dpp_max<0x111>(v);  // row_shr:1
    m = dpp_max<0x112>(m);
    if (NL > 4) m = dpp_max<0x114>(m);
    if (NL > 8) m = dpp_max<0x118>(m);
    if (NL > 16) {
        m = dpp_max<0x142>(m);  // row_bcast:15
        m = dpp_max<0x143>(m);  // row_bcast:31
    }
    m = lane_value(m, NL - 1);
    constexpr unsigned long long LN = NL == 64 ? ~0ull : (1ull << (NL & 63)) - 1;
    unsigned long long b = __ballot(x.i > 0 && v == m) & LN;
    if (b == 0) b = __ballot(x.i > 0) & LN;  // no number among the values
    if (b == 0) return VI{0.0, 0};
    int l = __builtin_ctzll(b);
    int i = __builtin_amdgcn_readlane(x.i, l);
    for (b &= b - 1; b; b &= b - 1) {
        const int l2 = __builtin_ctzll(b), i2 = __builtin_amdgcn_readlane(x.i, l2);
        if (i2 < i) { i = i2; l = l2; }
    }
    return VI{lane_value(x.v, l), i};
}
// Over the block of NW (up to 16) wavefronts with one barrier: successive calls alternate
// between the two halves of sh (4 NW entries; a half holds 2 NW so that the two-value form
// below shares them), so a call's writes never meet the previous call's reads and the
// trailing barrier that protects a single buffer is not needed.  tog is uniform over the
// block and flips on every call.
template <int NW>
__device__ __forceinline__ VI block_argmax_t(VI x, VI *sh, int &tog)
{
    const int tid = threadIdx.x;
    VI *b = sh + tog * 2 * NW;
    tog ^= 1;
    x = wave_argmax<64>(x);
    if ((tid & 63) == 0) b[tid >> 6] = x;
    __syncthreads();
    return wave_argmax<NW>(b[tid & (NW - 1)]);
}
// Two independent (value, index) maxima under one barrier, in the same alternating
// halves of sh.
template <int NW>
__device__ __forceinline__ void block_argmax2_t(VI &x, VI &y, VI *sh, int &tog)
{
    const int tid = threadIdx.x;
    VI *b = sh + tog * 2 * NW;
    tog ^= 1;
    x = wave_argmax<64>(x);
    y = wave_argmax<64>(y);
    if ((tid & 63) == 0) { b[tid >> 6] = x; b[NW + (tid >> 6)] = y; }
    __syncthreads();
    x = wave_argmax<NW>(b[tid & (NW - 1)]);
    y = wave_argmax<NW>(b[NW + (tid & (NW - 1))]);
}
// lanes per column of the swap check's scan: the k columns' rows are spread over all NTH
// threads, G (a power of two) to a column
__device__ __forceinline__ int scan_lanes(int k, int NTH)
{
    int g = 1;
    while (g < 64 && 2 * g * k <= NTH) g *= 2;
    return g;
}
// (value, smallest index) maximum over aligned groups of g lanes, the same in every lane of
// a group: values >= 0, a NaN counts as the smallest (compared as it is, it would stay in
// its own lane, and the lanes would go on with different columns)
__device__ __forceinline__ VI group_argmax(VI x, int g)
{
    if (!(x.v >= 0.0)) x.v = -1.0;
    if (g > 32) x = vi_step<32>(x);
    if (g > 16) x = vi_step<16>(x);
    if (g > 8) x = vi_step<8>(x);
    if (g > 4) x = vi_step<4>(x);
    if (g > 2) x = vi_step<2>(x);
    if (g > 1) x = vi_step<1>(x);
    return x;
}
// Orders a wavefront's own LDS accesses (it executes in lockstep; the fence completes
// its lanes' writes before any lane reads them)
__device__ __forceinline__ void wsync()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    __builtin_amdgcn_wave_barrier();
}
// x * t[0] * t[1] * ... * t[n - 1], multiplied in that order (one thread), with the
// factors read from LDS eight at a time ahead of their multiplications
__device__ __forceinline__ double ordered_prod(double x, const double *t, int n)
{
    int j = 0;
    for (; j + 8 <= n; j += 8) {
        double f[8];
        #pragma unroll
        for (int u = 0; u < 8; u++) f[u] = t[j + u];
        #pragma unroll
        for (int u = 0; u < 8; u++) x = x * f[u];
    }
    for (; j < n; j++) x = x * t[j];
    return x;
}

// ---------------------------------------------------------------------------
// leaf D blocks (CauchylikeEig on the leaf rows/cols, CauchyHssEig.f90:2089-2100)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(WG) void k_hss_dgen(const HssMerge *hm, const HssNode *nodes, int nn)
{
    int b = blockIdx.x;
    if (b >= nn) return;
    HssNode N = nodes[b];
    const HssMerge H = hm[N.mrg];
    int m = N.leaf_m, r0 = N.leaf_r0;  // leaf rows/cols r0+1 .. r0+m (1-based)
    double *out = H.dd + H.pd[N.node - 1];
    for (int e = threadIdx.x; e < m * m; e += WG) {
        int i = e % m, j = e / m;
        int pf = r0 + 1 + i, pw = r0 + 1 + j;
        double den = (pf <= pw) ? (A1(H.FF, pf) - A1(H.FF, pw)) - A1(H.DIFL, pw)
                                : (A1(H.FF, pf) - A1(H.FF, pw + 1)) - A1(H.DIFR, pw);
        if (H.sq) den = den * (A1(H.FF, pf) + A1(H.D0, pw));
        out[e] = A1(H.U0, pf) * A1(H.V0, pw) / den;
    }
    if (threadIdx.x == 0) H.dsz[N.node - 1] = m;
}

// inlined: a call would give the merge record an address, and the compiler would then
// keep it in scratch memory and reload its fields there inside the pivot steps
__device__ __forceinline__ long arena_take(const HssMerge &H, long n)
{
    unsigned long long o = atomicAdd(H.arena_top, (unsigned long long)n);
    if ((long)(o + n) > H.arena_cap) { atomicOr(H.err, 2); return -1; }
    return (long)o;
}
__device__ __forceinline__ long scratch_take(const HssMerge &H, long n)
{
    unsigned long long o = atomicAdd(H.scratch_top, (unsigned long long)n);
    if ((long)(o + n) > H.scratch_cap) { atomicOr(H.err, 4); return -1; }
    return (long)o;
}

// ---------------------------------------------------------------------------
// Row compression of one node: rrluCauchyEigrow + CauchylikeEigQ (ComprcauchyEig 'r')
// rows: the node's M row generators (LDS); columns: the N column generators
// outside the node (private copies: V in LDS when it fits, else global; PU global,
// with positions 1..min(M, N) mirrored in LDS).
// The passes over the N columns take HSS_RB = 2 columns per thread at a time: the loads of
// both (V, PU, then the roots' gathered values) are issued before any result is used, the
// next two's V and PU before the current results, and the stores after the loads.  The
// width is bounded by the code, not the registers: a step runs through four such passes
// and two searches, every one an inlined body, and with 7 columns (8 in the column
// compression) the kernels were 59-66 KB, as much as the instruction cache two CUs share
// (64 KB); with 2 they are 38-45 KB.  A pivot step of a node with 240 outside columns
// went from 17 to 11 thousand cycles, of one with 4000 from 33 to 27 thousand.  Widths 3
// and 4 are 1-3 % slower overall, 1024 threads 5-17 %, 256 threads 4-8 %; one wavefront
// for small nodes, without barriers, lost to the block once its reductions were short.
// A step the swap check does not follow runs the next step's row search inside its own
// row update and reduces it with the next step's first column search under one barrier.
// ---------------------------------------------------------------------------
template <int HSS_CWG, bool SQ>
__global__ __launch_bounds__(HSS_CWG) void k_hss_rowcomp(const HssMerge *hm, const HssNode *nodes, int nn,
                                                    double tol, int lds_cap)
{
    extern __shared__ double hss_dyn[];  // lds_cap doubles: V when the node's columns fit
    __shared__ double F[HSS_MAXM], A[HSS_MAXM], Z[HSS_MAXM], W[HSS_MAXM];
    // factors of the ordered products: W(k) on the last wavefront, the swap on thread 0
    __shared__ double T1[HSS_MAXM], T2[HSS_MAXM];
    __shared__ int PL[HSS_MAXM], PUs[HSS_MAXM];
    __shared__ short PQ[HSS_MAXM], IP[HSS_MAXM];   // positions within the node (<= HSS_MAXM)
    __shared__ VI red[4 * (HSS_CWG / 64)];
    int tog = 0;  // which half of red the next reduction uses
    __shared__ long s_off;
    __shared__ int s_M, s_N, s_Rk, s_flag, s_ii, s_jj;
    const int tid = threadIdx.x, lane = tid & 63;
    constexpr int RB = HSS_RB;
    if ((int)blockIdx.x >= nn) return;
    HssNode Nd = nodes[blockIdx.x];
    const HssMerge H = hm[Nd.mrg];
    int *lr = H.lr, *lc = H.lc;
    const int node = Nd.node;
    if (tid == 0) {
        if (Nd.c1 > 0) {
            lr[2 * (node - 1)] = lr[2 * (Nd.c1 - 1)]; lr[2 * (node - 1) + 1] = lr[2 * (Nd.c2 - 1) + 1];
            lc[2 * (node - 1)] = lc[2 * (Nd.c1 - 1)]; lc[2 * (node - 1) + 1] = lc[2 * (Nd.c2 - 1) + 1];
        }
        int M = lr[2 * (node - 1) + 1] - lr[2 * (node - 1)] + 1;
        int nic = lc[2 * (node - 1) + 1] - lc[2 * (node - 1)] + 1;
        s_M = M;
        s_N = *H.lca - nic;
        // a merge whose construction already failed is finished densely; skip it
        s_flag = (*H.err != 0 || M > HSS_MAXM || M < 1 || nic < 1 || s_N < 0) ? 1 : 0;
        s_off = s_flag ? -1 : scratch_take(H, 2L * (s_N > 0 ? s_N : 1));
        if (s_flag) atomicOr(H.err, 1);
    }
    __syncthreads();
    if (s_flag || s_off < 0) return;
    const int M = s_M, N = s_N, l0 = lr[2 * (node - 1)], c0 = lc[2 * (node - 1)], c1e = lc[2 * (node - 1) + 1];
    const int NS = N > 0 ? N : 1;
    const int mn = M < N ? M : N;
    // Private per column: the generator V (updated every step) and the root index PU;
    // the values of the root that its accurate differences read (FF, DIFL, DIFR and D0 at
    // PU and PU + 1) are shared by every node of the merge.  Kept in the dynamic LDS as
    // far as it holds them (lds_cap doubles): V; V and PU; or V, PU and the roots'
    // values, so that a small node's passes, swaps and pivot lookups stay in LDS.
    // Otherwise V and PU are global and the values are gathered by index.
    constexpr int RD = SQ ? 5 : 4;  // root values kept per column
    const bool vl = N <= lds_cap;   // all three uniform over the block
    const bool pl = (long)N + (N + 1) / 2 <= lds_cap;
    const bool sm = (long)N * (1 + RD) + (N + 1) / 2 <= lds_cap;
    constexpr int NTH = HSS_CWG;
    ldbl *Vl = (ldbl *)hss_dyn;
    ldbl *Rl = Vl + NS;  // sm: f0, f1, dl, dr (and s) of every column, NS apart
    __attribute__((address_space(3))) int *PUl =
        (__attribute__((address_space(3))) int *)(sm ? Rl + RD * NS : Vl + NS);
    gdblw *Vg = (gdblw *)(H.scratch + s_off);
    gint *PUg = (gint *)(H.scratch + s_off + NS);
    auto vld = [&](int j) -> double { return vl ? A1(Vl, j) : A1(Vg, j); };
    auto vst = [&](int j, double x) {
        if (vl) A1(Vl, j) = x;
        else A1(Vg, j) = x;
    };
    auto pu = [&](int j) -> int { return pl ? A1(PUl, j) : A1(PUg, j); };
    auto pu_set = [&](int j, int x) {
        if (pl) A1(PUl, j) = x;
        else A1(PUg, j) = x;
    };
    auto rl_get = [&](int j) -> RootG {
        return RootG{Rl[j - 1], Rl[NS + j - 1], Rl[2 * NS + j - 1], Rl[3 * NS + j - 1], SQ ? Rl[4 * NS + j - 1] : 0.0};
    };
    // the root values of the column at position j <= min(M, N)
    auto croot = [&](int j) -> RootG { return sm ? rl_get(j) : root_load<SQ>(H, A1(PUs, j)); };
    for (int j = tid; j < N; j += NTH) {
        int src = (j < c0 - 1) ? j + 1 : j + 1 + (c1e - c0 + 1);
        vst(j + 1, A1((gdbl *)H.V, src));
        const int p = A1((gcint *)H.PU, src);
        pu_set(j + 1, p);
        if (j < mn) PUs[j] = p;
        if (sm) {
            const RootG r = root_load<SQ>(H, p);
            Rl[j] = r.f0; Rl[NS + j] = r.f1; Rl[2 * NS + j] = r.dl; Rl[3 * NS + j] = r.dr;
            if (SQ) Rl[4 * NS + j] = r.s;
        }
    }
    // column swap (one thread; a barrier follows): every load before the first store, so
    // that their latencies overlap
    auto swapc = [&](int a, int c) {
        const double va = vld(a), vc = vld(c);
        const int u = pu(a), w = pu(c);
        double ra[RD], rc[RD];
        if (sm) {
            #pragma unroll
            for (int q = 0; q < RD; q++) { ra[q] = Rl[q * NS + a - 1]; rc[q] = Rl[q * NS + c - 1]; }
        }
        vst(a, vc); vst(c, va);
        pu_set(a, w); pu_set(c, u);
        if (a <= mn) A1(PUs, a) = w;
        if (c <= mn) A1(PUs, c) = u;
        if (sm) {
            #pragma unroll
            for (int q = 0; q < RD; q++) { Rl[q * NS + a - 1] = rc[q]; Rl[q * NS + c - 1] = ra[q]; }
        }
    };
    // row swap of the generators, likewise
    auto swapr = [&](int a, int c) {
        const double fa = A1(F, a), fc = A1(F, c), za = A1(Z, a), zc = A1(Z, c), aa = A1(A, a), ac = A1(A, c);
        const int la = A1(PL, a), lc2 = A1(PL, c);
        const short qa = A1(PQ, a), qc = A1(PQ, c);
        A1(F, a) = fc; A1(F, c) = fa;
        A1(Z, a) = zc; A1(Z, c) = za;
        A1(A, a) = ac; A1(A, c) = aa;
        A1(PL, a) = lc2; A1(PL, c) = la;
        A1(PQ, a) = qc; A1(PQ, c) = qa;
    };
    auto cload = [&](int j0, int *pw, double *v) {
        #pragma unroll
        for (int u = 0; u < RB; u++) {
            const int j = min(j0 + u * NTH, N);
            pw[u] = pu(j);
            v[u] = vld(j);
        }
    };
    // the columns' root values, from LDS or gathered
    auto rload = [&](int j0, const int *pw, RootG *c) {
        #pragma unroll
        for (int u = 0; u < RB; u++) c[u] = sm ? rl_get(min(j0 + u * NTH, N)) : root_load<SQ>(H, pw[u]);
    };
    // body(j, pw, v, c) for the columns j in [lo, N]; j may exceed N (loads clamped)
    auto cpass = [&](int lo, auto body) {
        int j0 = lo + tid;
        if (j0 > N) return;
        if (sm) {  // two columns at a time: their LDS loads and divides overlap
            for (int j = j0; j <= N; j += 2 * NTH) {
                const int p0 = A1(PUl, j);
                const double v0 = A1(Vl, j);
                const RootG c0r = rl_get(j);
                if (j - lane + NTH <= N) {  // uniform over the wavefront
                    const int j1 = min(j + NTH, N), p1 = A1(PUl, j1);
                    const double v1 = A1(Vl, j1);
                    const RootG c1r = rl_get(j1);
                    body(j, p0, v0, c0r);
                    body(j + NTH, p1, v1, c1r);
                } else {
                    body(j, p0, v0, c0r);
                }
            }
            return;
        }
        int pw[RB];
        double v[RB];
        cload(j0, pw, v);
        for (;;) {
            RootG c[RB];
            #pragma unroll
            for (int u = 0; u < RB; u++) c[u] = root_load<SQ>(H, pw[u]);
            const int jn = j0 + RB * NTH;
            int pn[RB];
            double vn[RB];
            if (jn <= N) cload(jn, pn, vn);
            #pragma unroll
            for (int u = 0; u < RB; u++) body(j0 + u * NTH, pw[u], v[u], c[u]);
            if (jn > N) break;
            j0 = jn;
            #pragma unroll
            for (int u = 0; u < RB; u++) { pw[u] = pn[u]; v[u] = vn[u]; }
        }
    };
    // max over j in [k, N] of |V(j) / fd(pd, PU(j))| (index j - k + 1), ffd = FF(pd)
    auto colsearch = [&](int k, int pd, double ffd) -> VI {
        VI y = {0.0, 0};
        cpass(k, [&](int j, int pw, double v, const RootG &c) {
            if (j <= N) y = vi_better(y, VI{fabs(v / fd_r<SQ>(ffd, pd, pw, c)), j - k + 1});
        });
        return y;
    };
    // max over i in [k, M] of |Z(i) / fd(PL(i), pw)|, w = the values of root pw
    auto rowsearch = [&](int k, int pw, const RootG &w) -> VI {
        VI x = {0.0, 0};
        for (int i = k + tid; i <= M; i += NTH)
            x = vi_better(x, VI{fabs(A1(Z, i) / fd_r<SQ>(A1(F, i), A1(PL, i), pw, w)), i - k + 1});
        return x;
    };
    // the same over the block's rows on every wavefront by itself: for few rows a second
    // or third pass over them costs less than a reduction over the block
    auto rowsearch_w = [&](int k, int pw, const RootG &w) -> VI {
        VI x = {0.0, 0};
        for (int i = k + lane; i <= M; i += 64)
            x = vi_better(x, VI{fabs(A1(Z, i) / fd_r<SQ>(A1(F, i), A1(PL, i), pw, w)), i - k + 1});
        return wave_argmax<64>(x);
    };
    for (int i = tid; i < M; i += NTH) {
        PL[i] = A1((gcint *)H.PL, l0 + i);
        A[i] = A1((gdbl *)H.U, l0 + i);
        F[i] = A1((gdbl *)H.FF, PL[i]);
        Z[i] = A[i];
        PQ[i] = (short)(i + 1);
        W[i] = 0.0;
    }
    __syncthreads();
    double amax = 0.0;
    int Rk = mn;
    const double rho = 1.5;
    bool pre = false;     // pre_cl, pre_rw hold this step's first row and column searches
    VI pre_cl = {0.0, 0}, pre_rw = {0.0, 0};
    RootG cnext = {0.0, 0.0, 0.0, 0.0, 0.0};  // root data of PU(k + 1) when pre
    // flop count of the reference's model (nflops of rrluCauchyEigrow and its pivot
    // searches, CauchyHssEig.f90:105, 147, 205, 680-703); the loop is uniform over the
    // block, thread 0 adds it to the merge's total
    unsigned long long fl = 0;
    for (int k = 1; k <= mn; k++) {
        // ---- CauchyPivtEig: rook search on the k-th Schur complement
        fl += 4ull * (M + N - 2 * k + 3);
        RootG cw;  // root data of the column at position k (PU(k)), kept through the step
        {
            VI cl, rw;
            if (pre) {
                cl = pre_cl;
                rw = pre_rw;
                cw = cnext;
            } else {
                const int pwk = A1(PUs, k);
                cw = croot(k);
                cl = rowsearch(k, pwk, cw);
                rw = colsearch(k, A1(PL, k), A1(F, k));
                block_argmax2_t<HSS_CWG / 64>(cl, rw, red, tog);
            }
            double junkL = cl.v * fabs(vld(k)), junkU = rw.v * fabs(A1(Z, k));
            double piv = fabs(A1(Z, k) * vld(k) / fd_r<SQ>(A1(F, k), A1(PL, k), A1(PUs, k), cw));
            if (!(junkL <= piv && junkU <= piv)) {
                int flg = (junkL > junkU) ? 1 : 0;
                int jjL = cl.i, jjU = rw.i;
                // Every thread has read position k for the tests above before any swap: a
                // row swap is made after the column search it feeds (which reads the
                // incoming row where it still is) and its reduction's barrier.
                if (flg == 0) __syncthreads();
                for (;;) {
                    if (flg == 1) {
                        const int jr = jjL + k - 1;
                        jjU = block_argmax_t<HSS_CWG / 64>(colsearch(k, A1(PL, jr), A1(F, jr)), red, tog).i;
                        fl += 4ull * (N - k + 1);
                        if (tid == 0) swapr(k, jr);
                        if (jjU == 1) {
                            __syncthreads();
                            break;
                        }
                    }
                    if (tid == 0) swapc(k, jjU + k - 1);
                    __syncthreads();
                    const int pwk2 = A1(PUs, k);
                    cw = croot(k);
                    const bool few = M - k < 256;
                    jjL = few ? rowsearch_w(k, pwk2, cw).i : block_argmax_t<HSS_CWG / 64>(rowsearch(k, pwk2, cw), red, tog).i;
                    fl += 4ull * (M - k + 1);
                    if (jjL == 1) {
                        if (few) __syncthreads();  // before the update pass writes what the search reads
                        break;
                    }
                    flg = 1;
                }
            }
        }
        // the search ended with a barrier after its last swap and its last reads (or made
        // none), so the update pass below may start without another
        double ukk = A1(Z, k) * vld(k) / fd_r<SQ>(A1(F, k), A1(PL, k), A1(PUs, k), cw);
        amax = fmax(amax, fabs(ukk));
        if (fabs(ukk) < tol * amax) {
            // ---- CauchyPivtEig_CP: complete pivoting over the Schur complement
            fl += 4ull * (M - k + 1) * (N - k + 1);
            VI best = {0.0, 0};
            VI bestrow = {0.0, 0};
            for (int j0 = k + tid; j0 <= N; j0 += RB * NTH) {
                int pw[RB];
                double v[RB], mv[RB];
                int mi[RB];
                RootG c[RB];
                cload(j0, pw, v);
                rload(j0, pw, c);
                #pragma unroll
                for (int u = 0; u < RB; u++) { mv[u] = -DBL_MAX; mi[u] = 0; }
                for (int i = k; i <= M; i++) {
                    const double zi = A1(Z, i), fi = A1(F, i);
                    const int pli = A1(PL, i);
                    #pragma unroll
                    for (int u = 0; u < RB; u++) {
                        const double den = fd_r<SQ>(fi, pli, pw[u], c[u]);
                        if (mi[u] != 0 && !may_exceed(zi, den, mv[u])) continue;
                        double vv = fabs(zi / den);
                        if (mi[u] == 0 || vv > mv[u]) { mv[u] = vv; mi[u] = i - k + 1; }
                    }
                }
                #pragma unroll
                for (int u = 0; u < RB; u++) {
                    const int j = j0 + u * NTH;
                    if (j > N) continue;
                    double jt = fabs(mv[u] * v[u]);
                    VI cc = {jt, j - k + 1};
                    VI nb = vi_better(best, cc);
                    if (nb.i == cc.i) bestrow.i = mi[u];
                    best = nb;
                }
            }
            VI win = block_argmax_t<HSS_CWG / 64>(best, red, tog);
            __syncthreads();
            if (win.i > 0 && best.i == win.i) { s_ii = bestrow.i; s_jj = win.i; }
            __syncthreads();
            if (tid == 0) {
                int ii = s_ii, jj = s_jj;
                swapr(k, ii + k - 1);
                swapc(k, jj + k - 1);
            }
            __syncthreads();
            cw = croot(k);
            ukk = A1(Z, k) * vld(k) / fd_r<SQ>(A1(F, k), A1(PL, k), A1(PUs, k), cw);
            amax = fmax(amax, fabs(ukk));
            if (fabs(ukk) < tol * amax) { Rk = k - 1; break; }
        }
        // ---- generator updates of the (k+1)-th Schur complement; unless a swap check
        // follows, the pass over the rows also runs step k+1's row search and the pass
        // over the columns its first column search
        const double Fk = A1(F, k);
        const int plk = A1(PL, k), puk = A1(PUs, k);
        const RootG ck = cw;
        const bool fuse = k + 1 <= mn && !(k % 10 == 0 && M - k > 0);
        const int fk1 = fuse ? A1(PL, k + 1) : 0;
        const double ff1 = fuse ? A1(F, k + 1) : 0.0;
        const int pun = fuse ? A1(PUs, k + 1) : puk;
        const RootG cn = fuse ? croot(k + 1) : cw;
        // The last wavefront updates W and forms W(k), an ordered product, while the others
        // are in their passes: its factors' gathers in parallel, then lane 0 multiplies.
        // W and T1 are touched by this wavefront alone until the barrier below.
        if (tid >= NTH - 64) {
            for (int j = k - 1 - lane; j >= 1; j -= 64) {
                double temp = -1.0 * fd_r<SQ>(A1(F, j), A1(PL, j), puk, ck);
                A1(W, j) = A1(W, j) * (temp / ppq<SQ>(Fk, A1(F, j)));
                const int puj = A1(PUs, j);
                const double t2 = -1.0 * fd_r<SQ>(Fk, plk, puj, croot(j));
                A1(T1, j) = t2 / ppq<SQ>(A1(F, j), Fk);
            }
            wsync();
            if (lane == 0) A1(W, k) = ordered_prod(fd_r<SQ>(Fk, plk, puk, ck) / A1(A, k), T1, k - 1);
        }
        VI x1 = {0.0, 0};
        for (int j = k + 1 + tid; j <= M; j += NTH) {
            double temp = fd_r<SQ>(A1(F, j), A1(PL, j), puk, ck);
            temp = ppq<SQ>(A1(F, j), Fk) / temp;
            const double zj = A1(Z, j) * temp;
            A1(Z, j) = zj;
            if (fuse) x1 = vi_better(x1, VI{fabs(zj / fd_r<SQ>(A1(F, j), A1(PL, j), pun, cn)), j - k});
        }
        VI y1 = {0.0, 0};
        cpass(k + 1, [&](int j, int pw, double v, const RootG &c) {
            double temp = dd_r<SQ>(pw, c, puk, ck);
            double temp2 = -1.0 * fd_r<SQ>(Fk, plk, pw, c);
            temp = temp / temp2;
            const double vj = v * temp;
            if (j <= N) {
                vst(j, vj);
                if (fuse) y1 = vi_better(y1, VI{fabs(vj / fd_r<SQ>(ff1, fk1, pw, c)), j - k});
            }
        });
        fl += 5ull * (M - k) + 7ull * (N - k) + 12ull * (k - 1);
        pre = fuse;
        // The reduction's barrier (or the one before a swap check) publishes the passes and W
        if (fuse) {
            block_argmax2_t<HSS_CWG / 64>(x1, y1, red, tog);
            pre_cl = x1;
            pre_rw = y1;
            cnext = cn;
        } else {
            __syncthreads();
        }
        // ---- every 10 steps: swap while max |Mat_N| > rho (searchMax2Eig)
        if (k % 10 == 0 && M - k > 0) {
            for (;;) {
                // per column the first largest entry over the rows, G lanes to a column (one
                // thread per column took 30-60 thousand cycles a check)
                VI x = {0.0, 0};
                const int G = scan_lanes(k, NTH), g = tid & (G - 1);
                for (int jc = 1 + tid / G; jc - tid / G <= k; jc += NTH / G) {
                    VI e = {0.0, 0};
                    if (jc <= k) {
                        const double fj = A1(F, jc);
                        for (int i = 1 + g; i <= M - k; i += G)
                            e = vi_better(e, VI{fabs(A1(Z, k + i) / ppq<SQ>(A1(F, k + i), fj)), i});
                    }
                    e = group_argmax(e, G);
                    if (jc <= k) {
                        const VI nb = vi_better(x, VI{e.v * fabs(A1(W, jc)), jc});
                        if (nb.i == jc && g == 0) IP[jc - 1] = (short)e.i;
                        x = nb;
                    }
                }
                VI win = block_argmax_t<HSS_CWG / 64>(x, red, tog);
                if (!(win.v > rho)) break;
                const int ii = win.i, jj = IP[ii - 1] + k;
                fl += 10ull * (N - k) + 8ull * M + 18ull * k;
                __syncthreads();
                const double Fii = A1(F, ii), Fjj = A1(F, jj);
                const int plii = A1(PL, ii), pljj = A1(PL, jj);
                cpass(k + 1, [&](int j, int pw, double v, const RootG &c) {
                    double temp = -1.0 * fd_r<SQ>(Fii, plii, pw, c);
                    double temp2 = -1.0 * fd_r<SQ>(Fjj, pljj, pw, c);
                    temp = temp / temp2;
                    if (j <= N) vst(j, v * temp);
                });
                for (int j = k + 1 + tid; j <= M; j += NTH) {
                    if (j == jj) continue;
                    A1(Z, j) = A1(Z, j) * (ppq<SQ>(A1(F, j), Fjj) / ppq<SQ>(A1(F, j), Fii));
                }
                for (int j = 1 + tid; j <= k; j += NTH) {
                    if (j == ii) continue;
                    A1(W, j) = A1(W, j) * (ppq<SQ>(A1(F, j), Fii) / ppq<SQ>(A1(F, j), Fjj));
                    const int puj = A1(PUs, j);
                    const RootG cj = croot(j);
                    double temp = fd_r<SQ>(Fii, plii, puj, cj);
                    A1(T1, j) = ppq<SQ>(Fii, A1(F, j)) / temp;
                    temp = -1.0 * fd_r<SQ>(Fjj, pljj, puj, cj);
                    A1(T2, j) = temp / ppq<SQ>(A1(F, j), Fjj);
                }
                __syncthreads();
                if (tid == 0) {
                    const int puii = A1(PUs, ii);
                    const RootG cii = croot(ii);
                    double uj = A1(A, ii) * (ppq<SQ>(Fii, Fjj) / fd_r<SQ>(Fii, plii, puii, cii));
                    double wi = fd_r<SQ>(Fjj, pljj, puii, cii) / A1(A, jj);
                    for (int j = 1; j <= k; j++) {
                        if (j == ii) continue;
                        uj = uj * A1(T1, j);
                        wi = wi * A1(T2, j);
                    }
                    A1(Z, jj) = uj;
                    A1(W, ii) = wi;
                    int u = A1(PL, ii); A1(PL, ii) = A1(PL, jj); A1(PL, jj) = u;
                    short q = A1(PQ, ii); A1(PQ, ii) = A1(PQ, jj); A1(PQ, jj) = q;
                    double t = A1(F, ii); A1(F, ii) = A1(F, jj); A1(F, jj) = t;
                    t = A1(A, ii); A1(A, ii) = A1(A, jj); A1(A, jj) = t;
                }
                __syncthreads();
            }
        }
    }
    // ---- U generator (CauchylikeEigQ, then rows back to the node order)
    for (int i = 1 + tid; i <= M; i += NTH) IP[A1(PQ, i) - 1] = (short)i;  // invp
    if (tid == 0) {
        atomicAdd(H.flops, fl);
        int r = Rk;
        if (r < mn) {
            s_Rk = r;
            s_off = arena_take(H, (long)M * (r > 0 ? r : 1));
        } else {
            s_Rk = M;
            s_off = arena_take(H, (long)M * M);
        }
        H.usz[2 * (node - 1)] = M;
        H.usz[2 * (node - 1) + 1] = s_Rk;
        H.pu[node - 1] = s_off;
    }
    __syncthreads();
    const long off = s_off;
    if (off >= 0) {
        double *Ug = H.arena + off;
        const int r = s_Rk;
        if (Rk < mn) {
            for (int e = tid; e < M * r; e += NTH) {
                int i = e % M + 1, j = e / M + 1;
                int src = IP[i - 1];  // row src of Q
                double q;
                if (src <= r) q = (src == j) ? 1.0 : 0.0;
                else q = A1(Z, src) * A1(W, j) / ppq<SQ>(A1(F, src), A1(F, j));
                Ug[e] = q;
            }
        } else {
            for (int e = tid; e < M * M; e += NTH) {
                int i = e % M + 1, j = e / M;
                Ug[e] = (IP[i - 1] - 1 == j) ? 1.0 : 0.0;
            }
        }
    }
    // permuted row generators and their indices back to the compacted arrays
    for (int i = tid; i < M; i += NTH) {
        A1(H.U, l0 + i) = A[i];
        A1(H.PL, l0 + i) = PL[i];
    }
}

// ---------------------------------------------------------------------------
// Column compression of one node: rrluCauchyEigcol + CauchylikeEigQ2
// (ComprcauchyEig 'c').  RRLU rows: the node's M columns (roots, alpha, LDS);
// RRLU columns: the N row generators outside the node (private copies, as in the row
// compression; their passes, the mirrored positions 1..min(M, N) and the fused next
// row search work the same way).
// ---------------------------------------------------------------------------
template <int HSS_CWG, bool SQ>
__global__ __launch_bounds__(HSS_CWG) void k_hss_colcomp(const HssMerge *hm, const HssNode *nodes, int nn,
                                                    double tol, int lds_cap)
{
    extern __shared__ double hss_dyn[];  // lds_cap doubles: V when the node's rows fit
    __shared__ double Dr[HSS_MAXM], A[HSS_MAXM], Z[HSS_MAXM], W[HSS_MAXM];
    // factors of the ordered products, as in the row compression; in the swap check the scanned
    // rows' root data
    __shared__ double T12[2 * HSS_MAXM];
    double *const T1 = T12, *const T2 = T12 + HSS_MAXM;
    __shared__ int PL[HSS_MAXM], PUs[HSS_MAXM];
    __shared__ short PQ[HSS_MAXM], IP[HSS_MAXM];   // positions within the node (<= HSS_MAXM)
    __shared__ VI red[4 * (HSS_CWG / 64)];
    int tog = 0;  // which half of red the next reduction uses
    __shared__ long s_off;
    __shared__ int s_M, s_N, s_Rk, s_flag, s_ii, s_jj;
    const int tid = threadIdx.x, lane = tid & 63;
    constexpr int RB = HSS_RB;
    if ((int)blockIdx.x >= nn) return;
    HssNode Nd = nodes[blockIdx.x];
    const HssMerge H = hm[Nd.mrg];
    int *lr = H.lr, *lc = H.lc;
    const int node = Nd.node;
    if (tid == 0) {
        int M = lc[2 * (node - 1) + 1] - lc[2 * (node - 1)] + 1;
        int nir = lr[2 * (node - 1) + 1] - lr[2 * (node - 1)] + 1;
        s_M = M;
        s_N = *H.lda - nir;
        s_flag = (*H.err != 0 || M > HSS_MAXM || M < 1 || nir < 1 || s_N < 0) ? 1 : 0;
        s_off = s_flag ? -1 : scratch_take(H, 2L * (s_N > 0 ? s_N : 1));
        if (s_flag) atomicOr(H.err, 1);
    }
    __syncthreads();
    if (s_flag || s_off < 0) return;
    const int M = s_M, N = s_N, c0 = lc[2 * (node - 1)], r0 = lr[2 * (node - 1)], r1e = lr[2 * (node - 1) + 1];
    const int mn = M < N ? M : N;
    // Private per outside row: its generator V (updated every step), pole index PU and
    // pole value FF(PU).  Kept in the dynamic LDS as far as it holds them: V; V and PU;
    // or V, PU, the pole values and the root values of the node's own M columns (FF,
    // DIFL, DIFR and D0 at PL and PL + 1), so that a small node's passes, swaps and row
    // searches stay in LDS.  Otherwise V and PU are global and the values gathered.
    constexpr int RD = SQ ? 5 : 4;
    gdbl *FF = (gdbl *)H.FF;
    const int NS = N > 0 ? N : 1;
    const bool vl = N <= lds_cap;  // all three uniform over the block
    const bool pl = (long)N + (N + 1) / 2 <= lds_cap;
    const bool sm = 2L * N + (N + 1) / 2 + (long)RD * M <= lds_cap;
    constexpr int NTH = HSS_CWG;
    ldbl *Vl = (ldbl *)hss_dyn;
    ldbl *FFl = Vl + NS;     // sm: FF(PU(j))
    ldbl *RRl = FFl + NS;    // sm: f0, f1, dl, dr (and s) of the node's M columns, M apart
    __attribute__((address_space(3))) int *PUl =
        (__attribute__((address_space(3))) int *)(sm ? RRl + RD * M : Vl + NS);
    gdblw *Vg = (gdblw *)(H.scratch + s_off);
    gint *PUg = (gint *)(H.scratch + s_off + NS);
    auto vld = [&](int j) -> double { return vl ? A1(Vl, j) : A1(Vg, j); };
    auto vst = [&](int j, double x) {
        if (vl) A1(Vl, j) = x;
        else A1(Vg, j) = x;
    };
    auto pu = [&](int j) -> int { return pl ? A1(PUl, j) : A1(PUg, j); };
    auto pu_set = [&](int j, int x) {
        if (pl) A1(PUl, j) = x;
        else A1(PUg, j) = x;
    };
    // the root values of the node's column at position i (PL(i))
    auto rroot = [&](int i) -> RootG {
        if (sm)
            return RootG{RRl[i - 1], RRl[M + i - 1], RRl[2 * M + i - 1], RRl[3 * M + i - 1],
                         SQ ? RRl[4 * M + i - 1] : 0.0};
        return root_load<SQ>(H, A1(PL, i));
    };
    for (int j = tid; j < N; j += NTH) {
        int src = (j < r0 - 1) ? j + 1 : j + 1 + (r1e - r0 + 1);
        vst(j + 1, A1((gdbl *)H.U, src));
        const int p = A1((gcint *)H.PL, src);
        pu_set(j + 1, p);
        if (j < mn) PUs[j] = p;
        if (sm) FFl[j] = A1(FF, p);
    }
    // outside-row swap (one thread; a barrier follows)
    auto swapc = [&](int a, int c) {
        const double va = vld(a), vc = vld(c);
        const int u = pu(a), w = pu(c);
        const double fa = sm ? A1(FFl, a) : 0.0, fc = sm ? A1(FFl, c) : 0.0;
        vst(a, vc); vst(c, va);
        pu_set(a, w); pu_set(c, u);
        if (a <= mn) A1(PUs, a) = w;
        if (c <= mn) A1(PUs, c) = u;
        if (sm) { A1(FFl, a) = fc; A1(FFl, c) = fa; }
    };
    // node-column swap of Dr, A, PL, PQ and the root values; of Z too unless the swap check
    // replaces Z (zs)
    auto swapr = [&](int a, int c, bool zs) {
        const double da = A1(Dr, a), dc = A1(Dr, c), za = A1(Z, a), zc = A1(Z, c), aa = A1(A, a), ac = A1(A, c);
        const int la = A1(PL, a), lc2 = A1(PL, c);
        const short qa = A1(PQ, a), qc = A1(PQ, c);
        double ra[RD], rc[RD];
        if (sm) {
            #pragma unroll
            for (int q = 0; q < RD; q++) { ra[q] = RRl[q * M + a - 1]; rc[q] = RRl[q * M + c - 1]; }
        }
        A1(Dr, a) = dc; A1(Dr, c) = da;
        if (zs) { A1(Z, a) = zc; A1(Z, c) = za; }
        A1(A, a) = ac; A1(A, c) = aa;
        A1(PL, a) = lc2; A1(PL, c) = la;
        A1(PQ, a) = qc; A1(PQ, c) = qa;
        if (sm) {
            #pragma unroll
            for (int q = 0; q < RD; q++) { RRl[q * M + a - 1] = rc[q]; RRl[q * M + c - 1] = ra[q]; }
        }
    };
    auto cload = [&](int j0, int *pd, double *v) {
        #pragma unroll
        for (int u = 0; u < RB; u++) {
            const int j = min(j0 + u * NTH, N);
            pd[u] = pu(j);
            v[u] = vld(j);
        }
    };
    auto fload = [&](int j0, const int *pd, double *ffd) {
        #pragma unroll
        for (int u = 0; u < RB; u++) ffd[u] = sm ? A1(FFl, min(j0 + u * NTH, N)) : A1(FF, pd[u]);
    };
    // body(j, pd, v, FF(pd)) for the outside rows j in [lo, N]; j may exceed N
    auto cpass = [&](int lo, auto body) {
        int j0 = lo + tid;
        if (j0 > N) return;
        if (sm) {  // two rows at a time: their LDS loads and divides overlap
            for (int j = j0; j <= N; j += 2 * NTH) {
                const int p0 = A1(PUl, j);
                const double v0 = A1(Vl, j), f0 = A1(FFl, j);
                if (j - lane + NTH <= N) {  // uniform over the wavefront
                    const int j1 = min(j + NTH, N), p1 = A1(PUl, j1);
                    const double v1 = A1(Vl, j1), f1 = A1(FFl, j1);
                    body(j, p0, v0, f0);
                    body(j + NTH, p1, v1, f1);
                } else {
                    body(j, p0, v0, f0);
                }
            }
            return;
        }
        int pd[RB];
        double v[RB];
        cload(j0, pd, v);
        for (;;) {
            double ffd[RB];
            #pragma unroll
            for (int u = 0; u < RB; u++) ffd[u] = A1(FF, pd[u]);
            const int jn = j0 + RB * NTH;
            int pn[RB];
            double vn[RB];
            if (jn <= N) cload(jn, pn, vn);
            #pragma unroll
            for (int u = 0; u < RB; u++) body(j0 + u * NTH, pd[u], v[u], ffd[u]);
            if (jn > N) break;
            j0 = jn;
            #pragma unroll
            for (int u = 0; u < RB; u++) { pd[u] = pn[u]; v[u] = vn[u]; }
        }
    };
    // max over j in [k, N] of |V(j) / fd(PU(j), pw)| (index j - k + 1), w = root values of pw
    auto colsearch = [&](int k, int pw, const RootG &w) -> VI {
        VI y = {0.0, 0};
        cpass(k, [&](int j, int pd, double v, double ffd) {
            if (j <= N) y = vi_better(y, VI{fabs(v / fd_r<SQ>(ffd, pd, pw, w)), j - k + 1});
        });
        return y;
    };
    // max over i in [k, M] of |Z(i) / fd(pd, PL(i))|, ffd = FF(pd)
    auto rowsearch = [&](int k, int pd, double ffd) -> VI {
        VI x = {0.0, 0};
        for (int i = k + tid; i <= M; i += NTH)
            x = vi_better(x, VI{fabs(A1(Z, i) / fd_r<SQ>(ffd, pd, A1(PL, i), rroot(i))), i - k + 1});
        return x;
    };
    // the same on every wavefront by itself, as in the row compression
    auto rowsearch_w = [&](int k, int pd, double ffd) -> VI {
        VI x = {0.0, 0};
        for (int i = k + lane; i <= M; i += 64)
            x = vi_better(x, VI{fabs(A1(Z, i) / fd_r<SQ>(ffd, pd, A1(PL, i), rroot(i))), i - k + 1});
        return wave_argmax<64>(x);
    };
    for (int i = tid; i < M; i += NTH) {
        Dr[i] = A1((gdbl *)H.D, c0 + i);
        A[i] = A1((gdbl *)H.V, c0 + i);
        PL[i] = A1((gcint *)H.PU, c0 + i);
        Z[i] = A[i];
        PQ[i] = (short)(i + 1);
        W[i] = 0.0;
        if (sm) {
            const RootG r = root_load<SQ>(H, PL[i]);
            RRl[i] = r.f0; RRl[M + i] = r.f1; RRl[2 * M + i] = r.dl; RRl[3 * M + i] = r.dr;
            if (SQ) RRl[4 * M + i] = r.s;
        }
    }
    __syncthreads();
    double amax = 0.0;
    int Rk = mn;
    const double rho = 1.5;
    bool pre = false;     // pre_cl, pre_rw hold this step's first row and column searches
    VI pre_cl = {0.0, 0}, pre_rw = {0.0, 0};
    RootG cnext = {0.0, 0.0, 0.0, 0.0, 0.0};  // root data of PL(k + 1) when pre
    double ffnext = 0.0;                      // FF(PU(k + 1)) when pre
    // flop count of the reference's model (rrluCauchyEigcol, CauchyHssEig.f90:321, 371,
    // 460, and its pivot searches), added to the merge's total by thread 0
    unsigned long long fl = 0;
    for (int k = 1; k <= mn; k++) {
        // ---- CauchyPivtEigm
        fl += 4ull * (M + N - 2 * k + 3);
        RootG cr;    // root data of PL(k), kept through the step
        double ffp;  // FF(PU(k)), kept through the step
        {
            VI cl, rw;
            if (pre) {
                cl = pre_cl;
                rw = pre_rw;
                cr = cnext;
                ffp = ffnext;
            } else {
                const int puk = A1(PUs, k), plk = A1(PL, k);
                ffp = A1(FF, puk);
                cr = rroot(k);
                cl = rowsearch(k, puk, ffp);
                rw = colsearch(k, plk, cr);
                block_argmax2_t<HSS_CWG / 64>(cl, rw, red, tog);
            }
            double junkL = cl.v * fabs(vld(k)), junkU = rw.v * fabs(A1(Z, k));
            double den;
            {
                const int plk = A1(PL, k), puk = A1(PUs, k);
                if (plk < puk) den = (cr.f1 - ffp) + cr.dr;
                else den = (cr.f0 - ffp) + cr.dl;
                if (SQ) den = den * (cr.s + ffp);
            }
            double piv = fabs(A1(Z, k) * vld(k) / den);
            if (!(junkL <= piv && junkU <= piv)) {
                int flg = (junkL > junkU) ? 1 : 0;
                int jjL = cl.i, jjU = rw.i;
                // barriers as in the row compression
                if (flg == 0) __syncthreads();
                for (;;) {
                    if (flg == 1) {
                        const int jr = jjL + k - 1;
                        const int plr = A1(PL, jr);
                        cr = rroot(jr);
                        jjU = block_argmax_t<HSS_CWG / 64>(colsearch(k, plr, cr), red, tog).i;
                        fl += 4ull * (N - k + 1);
                        if (tid == 0) swapr(k, jr, true);
                        if (jjU == 1) {
                            __syncthreads();
                            break;
                        }
                    }
                    if (tid == 0) swapc(k, jjU + k - 1);
                    __syncthreads();
                    const int puk2 = A1(PUs, k);
                    ffp = A1(FF, puk2);
                    const bool few = M - k < 256;
                    jjL = few ? rowsearch_w(k, puk2, ffp).i : block_argmax_t<HSS_CWG / 64>(rowsearch(k, puk2, ffp), red, tog).i;
                    fl += 4ull * (M - k + 1);
                    if (jjL == 1) {
                        if (few) __syncthreads();  // before the update pass writes what the search reads
                        break;
                    }
                    flg = 1;
                }
            }
        }
        // the search ended with a barrier, as in the row compression
        double ukk = A1(Z, k) * vld(k) / (-1.0 * fd_r<SQ>(ffp, A1(PUs, k), A1(PL, k), cr));
        amax = fmax(amax, fabs(ukk));
        if (fabs(ukk) < tol * amax) {
            // ---- CauchyPivtEigm_CP
            fl += 4ull * (M - k + 1) * (N - k + 1);
            VI best = {0.0, 0};
            int bestrow = 0;
            for (int j0 = k + tid; j0 <= N; j0 += RB * NTH) {
                int pd[RB];
                double v[RB], ffd[RB], mv[RB];
                int mi[RB];
                cload(j0, pd, v);
                fload(j0, pd, ffd);
                #pragma unroll
                for (int u = 0; u < RB; u++) { mv[u] = 0.0; mi[u] = 0; }
                for (int i = k; i <= M; i++) {
                    const double zi = A1(Z, i);
                    const int pli = A1(PL, i);
                    const RootG ri = rroot(i);
                    #pragma unroll
                    for (int u = 0; u < RB; u++) {
                        const double den = fd_r<SQ>(ffd[u], pd[u], pli, ri);
                        if (mi[u] != 0 && !may_exceed(zi, den, mv[u])) continue;
                        double vv = fabs(zi / den);
                        if (mi[u] == 0 || vv > mv[u]) { mv[u] = vv; mi[u] = i - k + 1; }
                    }
                }
                #pragma unroll
                for (int u = 0; u < RB; u++) {
                    const int j = j0 + u * NTH;
                    if (j > N) continue;
                    VI c = {fabs(mv[u] * v[u]), j - k + 1};
                    VI nb = vi_better(best, c);
                    if (nb.i == c.i) bestrow = mi[u];
                    best = nb;
                }
            }
            VI win = block_argmax_t<HSS_CWG / 64>(best, red, tog);
            if (win.i > 0 && best.i == win.i) { s_ii = bestrow; s_jj = win.i; }
            __syncthreads();
            if (tid == 0) {
                swapr(k, s_ii + k - 1, true);
                swapc(k, s_jj + k - 1);
            }
            __syncthreads();
            cr = rroot(k);
            ffp = A1(FF, A1(PUs, k));
            ukk = A1(Z, k) * vld(k) / (-1.0 * fd_r<SQ>(ffp, A1(PUs, k), A1(PL, k), cr));
            amax = fmax(amax, fabs(ukk));
            if (fabs(ukk) < tol * amax) { Rk = k - 1; break; }
        }
        const int plk = A1(PL, k), puk = A1(PUs, k);
        const double Fk = ffp;
        const RootG ck = cr;
        const bool fuse = k + 1 <= mn && !(k % 10 == 0 && M - k > 0);
        const int plk1 = fuse ? A1(PL, k + 1) : plk;
        const int pun = fuse ? A1(PUs, k + 1) : puk;
        const RootG ck1 = fuse ? rroot(k + 1) : ck;
        const double ffn = A1(FF, pun);
        // W on the last wavefront, as in the row compression
        if (tid >= NTH - 64) {
            for (int j = k - 1 - lane; j >= 1; j -= 64) {
                const int plj = A1(PL, j), puj = A1(PUs, j);
                const RootG rj = rroot(j);
                double temp = fd_r<SQ>(Fk, puk, plj, rj);
                double temp2 = dd_r<SQ>(plk, ck, plj, rj);
                temp = temp / temp2;
                A1(W, j) = A1(W, j) * temp;
                temp = fd_r<SQ>(sm ? A1(FFl, j) : A1(FF, puj), puj, plk, ck);
                temp2 = dd_r<SQ>(plj, rj, plk, ck);
                A1(T1, j) = temp / temp2;
            }
            wsync();
            if (lane == 0) A1(W, k) = ordered_prod((-1.0 * fd_r<SQ>(Fk, puk, plk, ck)) / A1(A, k), T1, k - 1);
        }
        VI x1 = {0.0, 0};
        for (int j = k + 1 + tid; j <= M; j += NTH) {
            const int plj = A1(PL, j);
            const RootG rj = rroot(j);
            double temp = dd_r<SQ>(plj, rj, plk, ck);
            double temp2 = -1.0 * fd_r<SQ>(Fk, puk, plj, rj);
            temp = temp / temp2;
            const double zj = A1(Z, j) * temp;
            A1(Z, j) = zj;
            if (fuse) x1 = vi_better(x1, VI{fabs(zj / fd_r<SQ>(ffn, pun, plj, rj)), j - k});
        }
        VI y1 = {0.0, 0};
        cpass(k + 1, [&](int j, int pd, double v, double ffd) {
            double temp = fd_r<SQ>(ffd, pd, plk, ck);
            const double vj = v * (ppq<SQ>(ffd, Fk) / temp);
            if (j <= N) {
                vst(j, vj);
                if (fuse) y1 = vi_better(y1, VI{fabs(vj / fd_r<SQ>(ffd, pd, plk1, ck1)), j - k});
            }
        });
        fl += 6ull * (M - k) + 5ull * (N - k) + 14ull * (k - 1);
        pre = fuse;
        // the barrier publishes the passes and W
        if (fuse) {
            block_argmax2_t<HSS_CWG / 64>(x1, y1, red, tog);
            pre_cl = x1;
            pre_rw = y1;
            cnext = ck1;
            ffnext = ffn;
        } else {
            __syncthreads();
        }
        if (k % 10 == 0 && M - k > 0) {
            for (;;) {
                // the scanned rows' root data, gathered once into T1 / T2 when they fit
                const int L = M - k;
                const bool stg = !sm && L * (SQ ? 5 : 4) <= 2 * HSS_MAXM;
                if (stg) {
                    for (int q = tid; q < L; q += NTH) {
                        const RootG r = root_load<SQ>(H, A1(PL, k + 1 + q));
                        T12[q] = r.f0;
                        T12[L + q] = r.f1;
                        T12[2 * L + q] = r.dl;
                        T12[3 * L + q] = r.dr;
                        if (SQ) T12[4 * L + q] = r.s;
                    }
                    __syncthreads();
                }
                VI x = {0.0, 0};
                const int G = scan_lanes(k, NTH), g = tid & (G - 1);  // as in the row compression
                for (int jc = 1 + tid / G; jc - tid / G <= k; jc += NTH / G) {
                    VI e = {0.0, 0};
                    if (jc <= k) {
                        const int pljc = A1(PL, jc);
                        const RootG rc = rroot(jc);
                        for (int i = 1 + g; i <= L; i += G) {
                            double tt;
                            if (sm) {
                                tt = dd_r<SQ>(A1(PL, i + k), rroot(i + k), pljc, rc);
                            } else if (stg) {
                                const RootG ri = {T12[i - 1], T12[L + i - 1], T12[2 * L + i - 1], T12[3 * L + i - 1],
                                                  SQ ? T12[4 * L + i - 1] : 0.0};
                                tt = dd_r<SQ>(A1(PL, i + k), ri, pljc, rc);
                            } else {
                                tt = ddq<SQ>(H, A1(PL, i + k), pljc);
                            }
                            e = vi_better(e, VI{fabs(A1(Z, k + i) / tt), i});
                        }
                    }
                    e = group_argmax(e, G);
                    if (jc <= k) {
                        const VI nb = vi_better(x, VI{e.v * fabs(A1(W, jc)), jc});
                        if (nb.i == jc && g == 0) IP[jc - 1] = (short)e.i;
                        x = nb;
                    }
                }
                VI win = block_argmax_t<HSS_CWG / 64>(x, red, tog);
                if (!(win.v > rho)) break;
                const int ii = win.i, jj = IP[ii - 1] + k;
                fl += 10ull * (N - k) + 12ull * M + 22ull * k;
                __syncthreads();
                const int plii = A1(PL, ii), pljj = A1(PL, jj);
                const RootG cii = rroot(ii), cjj = rroot(jj);
                cpass(k + 1, [&](int j, int pd, double v, double ffd) {
                    double temp = fd_r<SQ>(ffd, pd, plii, cii);
                    double temp2 = fd_r<SQ>(ffd, pd, pljj, cjj);
                    temp = temp / temp2;
                    if (j <= N) vst(j, v * temp);
                });
                for (int j = k + 1 + tid; j <= M; j += NTH) {
                    if (j == jj) continue;
                    double temp = ddq<SQ>(H, A1(PL, j), pljj);
                    double temp2 = ddq<SQ>(H, A1(PL, j), plii);
                    temp = temp / temp2;
                    A1(Z, j) = A1(Z, j) * temp;
                }
                for (int j = 1 + tid; j <= k; j += NTH) {
                    if (j == ii) continue;
                    const int puj = A1(PUs, j);
                    double temp = ddq<SQ>(H, A1(PL, j), plii);
                    double temp2 = ddq<SQ>(H, A1(PL, j), pljj);
                    temp = temp / temp2;
                    A1(W, j) = A1(W, j) * temp;
                    temp = ddq<SQ>(H, plii, A1(PL, j));
                    temp2 = -1.0 * fdq<SQ>(H, puj, plii);
                    A1(T1, j) = temp / temp2;
                    temp = fdq<SQ>(H, puj, pljj);
                    temp2 = ddq<SQ>(H, A1(PL, j), pljj);
                    A1(T2, j) = temp / temp2;
                }
                __syncthreads();
                if (tid == 0) {
                    const int puii = A1(PUs, ii);
                    double temp = ddq<SQ>(H, plii, pljj);
                    double temp2 = -1.0 * fdq<SQ>(H, puii, plii);
                    double uj = A1(A, ii) * (temp / temp2);
                    double wi = (-1.0 * fdq<SQ>(H, puii, pljj)) / A1(A, jj);
                    for (int j = 1; j <= k; j++) {
                        if (j == ii) continue;
                        uj = uj * A1(T1, j);
                        wi = wi * A1(T2, j);
                    }
                    A1(Z, jj) = uj;
                    A1(W, ii) = wi;
                    swapr(ii, jj, false);
                }
                __syncthreads();
            }
        }
    }
    // ---- V generator (CauchylikeEigQ2, columns back to the node order)
    for (int i = 1 + tid; i <= M; i += NTH) IP[A1(PQ, i) - 1] = (short)i;  // invp
    if (tid == 0) {
        atomicAdd(H.flops, fl);
        if (Rk < mn) {
            s_Rk = Rk;
            s_off = arena_take(H, (long)(Rk > 0 ? Rk : 1) * M);
        } else {
            s_Rk = M;
            s_off = arena_take(H, (long)M * M);
        }
        H.vsz[2 * (node - 1)] = s_Rk;
        H.vsz[2 * (node - 1) + 1] = M;
        H.pv[node - 1] = s_off;
    }
    __syncthreads();
    const long off = s_off;
    if (off >= 0) {
        double *Vg = H.arena + off;
        const int r = s_Rk;
        if (Rk < mn) {
            for (int e = tid; e < r * M; e += NTH) {
                int i = e % r + 1, j = e / r + 1;
                int src = IP[j - 1];  // column src of Q
                double q;
                if (src <= r) {
                    q = (src == i) ? 1.0 : 0.0;
                } else {
                    int pdjj = A1(PL, src), pdii = A1(PL, i);
                    double den;
                    if (pdii < pdjj) den = (A1(H.FF, pdii + 1) - A1(H.FF, pdjj)) + (A1(H.DIFR, pdii) - A1(H.DIFL, pdjj));
                    else den = (A1(H.FF, pdii) - A1(H.FF, pdjj + 1)) + (A1(H.DIFL, pdii) - A1(H.DIFR, pdjj));
                    if (SQ) den = den * (A1(H.D0, pdii) + A1(H.D0, pdjj));
                    q = -1.0 * A1(W, i) * A1(Z, src) / den;
                }
                Vg[e] = q;
            }
        } else {
            for (int e = tid; e < M * M; e += NTH) {
                int i = e % M, j = e / M + 1;
                Vg[e] = (IP[j - 1] - 1 == i) ? 1.0 : 0.0;
            }
        }
    }
    for (int i = tid; i < M; i += NTH) {
        A1(H.D, c0 + i) = Dr[i];
        A1(H.V, c0 + i) = A[i];
        A1(H.PU, c0 + i) = PL[i];
    }
}

// ---------------------------------------------------------------------------
// Compaction after a level (one block per merge): keep the first rank entries of
// every node of the level, then the full ranges of shallower leaves, in order.
// rows: U/PL with usz(2,:); cols: V/D/PU with vsz(1,:).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(WG) void k_hss_compact(const HssMerge *hm, const HssCompact *cp, const int *order,
                                                    int rows)
{
    // Every node's count and source start read in parallel, one thread per node; the
    // start of each node's slice by a prefix over LDS; then one pass over all elements,
    // each finding its node by binary search over the slice starts.
    __shared__ int s_start[1024 + 1], s_src[1024];
    HssCompact C = cp[blockIdx.x];
    const HssMerge H = hm[C.mrg];
    const int tid = threadIdx.x;
    int *rng = rows ? H.lr : H.lc;
    if (tid == 0) *H.scratch_top = 0ULL;  // the next compression starts its private copies afresh
    if (*H.err) return;
    // the host builds trees of at most 512 leaves, so a compaction lists at most 1024
    // nodes; a larger one would not fit the slice table and sends the merge dense
    if (C.count > 1024) {
        if (tid == 0) atomicOr(H.err, 1);
        return;
    }
    for (int q = tid; q < C.count; q += WG) {
        const int nd = order[C.start + q];
        const int r0 = rng[2 * (nd - 1)], have = rng[2 * (nd - 1) + 1] - r0 + 1;
        int cnt = have;
        if (q < C.nlevel) cnt = rows ? H.usz[2 * (nd - 1) + 1] : H.vsz[2 * (nd - 1)];
        if (cnt < 0 || cnt > have) cnt = 0;
        s_start[q] = cnt;
        s_src[q] = r0;  // 1-based
    }
    __syncthreads();
    if (tid == 0) {
        int lt = 0;
        for (int q = 0; q < C.count; q++) {
            const int c = s_start[q];
            s_start[q] = lt;
            lt += c;
        }
        s_start[C.count] = lt;
    }
    __syncthreads();
    double *Td = H.T, *Td2 = H.T + H.K;
    int *Ti = (int *)(H.T + 2 * H.K);
    const int tot = s_start[C.count];
    for (int d = tid; d < tot; d += WG) {
        int lo = 0, hi = C.count - 1;
        while (lo < hi) {
            const int md = (lo + hi + 1) >> 1;
            if (s_start[md] <= d) lo = md;
            else hi = md - 1;
        }
        const int sidx = s_src[lo] + (d - s_start[lo]);
        if (rows) { Td[d] = A1(H.U, sidx); Ti[d] = A1(H.PL, sidx); }
        else { Td[d] = A1(H.V, sidx); Td2[d] = A1(H.D, sidx); Ti[d] = A1(H.PU, sidx); }
    }
    __syncthreads();
    for (int d = tid; d < tot; d += WG) {
        if (rows) { H.U[d] = Td[d]; H.PL[d] = Ti[d]; }
        else { H.V[d] = Td[d]; H.D[d] = Td2[d]; H.PU[d] = Ti[d]; }
    }
    for (int q = tid; q < C.count; q += WG) {
        const int nd = order[C.start + q];
        rng[2 * (nd - 1)] = s_start[q] + 1;
        rng[2 * (nd - 1) + 1] = s_start[q + 1];
    }
    if (tid == 0) {
        if (rows) *H.lda = tot; else *H.lca = tot;
    }
}

// B generators of the nodes of one level: B_i = C(row skeleton of i, column
// skeleton of its sibling) (CauchyHssEig.f90:2229-2244).
__global__ __launch_bounds__(WG) void k_hss_bgen(const HssMerge *hm, const HssNode *nodes, int nn)
{
    __shared__ long s_off;
    if ((int)blockIdx.x >= nn) return;
    HssNode Nd = nodes[blockIdx.x];
    const HssMerge H = hm[Nd.mrg];
    const int node = Nd.node, sib = Nd.sib;
    const int r0 = H.lr[2 * (node - 1)], mi = H.lr[2 * (node - 1) + 1] - r0 + 1;
    const int c0 = H.lc[2 * (sib - 1)], nj = H.lc[2 * (sib - 1) + 1] - c0 + 1;
    if (*H.err || mi < 0 || nj < 0) return;
    if (threadIdx.x == 0) {
        s_off = arena_take(H, (long)mi * nj);
        H.bsz[2 * (node - 1)] = mi;
        H.bsz[2 * (node - 1) + 1] = nj;
        H.pb[node - 1] = s_off;
    }
    __syncthreads();
    if (s_off < 0) return;
    double *B = H.arena + s_off;
    for (int e = threadIdx.x; e < mi * nj; e += WG) {
        int i = e % mi, j = e / mi;
        int pf = A1(H.PL, r0 + i), pw = A1(H.PU, c0 + j);
        double fj = A1(H.FF, pw), vj = A1(H.V, c0 + j);
        double den = (pf <= pw) ? (A1(H.FF, pf) - fj) - A1(H.DIFL, pw)
                                : (A1(H.FF, pf) - A1(H.FF, pw + 1)) - A1(H.DIFR, pw);
        if (H.sq) den = den * (A1(H.FF, pf) + A1(H.D0, pw));
        B[e] = A1(H.U, r0 + i) * vj / den;
    }
}

// initial compacted arrays: D = roots, U = z, V = alpha, PL = PU = identity
__global__ __launch_bounds__(WG) void k_hss_init(const HssMerge *hm)
{
    const HssMerge H = hm[blockIdx.y];
    for (int i = blockIdx.x * WG + threadIdx.x; i < H.K; i += gridDim.x * WG) {
        H.D[i] = H.D0[i]; H.U[i] = H.U0[i]; H.V[i] = H.V0[i];
        H.PL[i] = i + 1; H.PU[i] = i + 1;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) { *H.lda = H.K; *H.lca = H.K; }
}

// ---------------------------------------------------------------------------
// Batched GEMM of the HSS multiply: work item (blockIdx.y) = one BG, block
// (blockIdx.x, blockIdx.z) = one 128 x 64 tile of its output.  FP64 MFMA 16x16x4.
// The k range is walked in chunks of 32: the block stages a 128 x 32 slab of A and
// a 32 x 64 slab of B in LDS (coalesced loads by all 256 threads), and while the
// four wavefronts multiply out of LDS the next chunk is already loading into
// registers.  Each wavefront owns 32 x 64 outputs in 8 accumulators; the k-steps
// of 4 run in order, as the single-product reference order of the tests expects.
// ---------------------------------------------------------------------------
typedef double d4h __attribute__((ext_vector_type(4)));
// The operand pointers of a BG are read from the item table, so the compiler cannot see
// that they point to global memory and would use FLAT loads, which count in LGKM_CNT as
// well as VM_CNT: every wait for the LDS operand reads would then also wait for the next
// chunk's loads.  Global-address-space views keep the two counters apart.
// what a staged element outside the operands reads
static __device__ double bg_zero = 0.0;
#define BG_BK 32
#define BG_AP 132  // LDS pitch of the A slab (128 rows + 4: no bank conflicts between k rows)
#define BG_BP 68   // LDS pitch of the B slab (64 columns + 4)
__global__ __launch_bounds__(WG) void k_bgemm(const BG *items)
{
    __shared__ double As[BG_BK * BG_AP];
    __shared__ double Bs[BG_BK * BG_BP];
    const BG g = items[blockIdx.y];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int rb = blockIdx.x * 128, c0 = blockIdx.z * 64;
    if (rb >= g.nrow || c0 >= g.n) return;  // the whole block
    const int K1 = g.k, K = g.k + g.k2;
    const long lda = g.lda, lda2 = g.lda2, ldb = g.ldb, ldb2 = g.ldb2;
    // staging of one chunk: A element (row rb + (i & 127), k kc + (i >> 7)), i = tid + 256 q;
    // B element i = tid + 256 q: (k kc + (i & 31), column c0 + (i >> 5)) column-major,
    // (k kc + (i >> 6), column c0 + (i & 63)) for btrans
    double ra[16], rbv[8];
    gdbl *const zero = (gdbl *)&bg_zero;  // unconditional global loads (k_bgemm_w)
    auto stage = [&](int kc) {
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const int i = tid + 256 * q, row = rb + (i & 127), t = kc + (i >> 7);
            const bool ok = row < g.nrow && t < K;
            gdbl *p = t < K1 ? (gdbl *)g.A + (row + (long)t * lda) : (gdbl *)g.A2 + (row + (long)(t - K1) * lda2);
            ra[q] = *(ok ? p : zero);
        }
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const int i = tid + 256 * q;
            int t, col;
            if (g.btrans) { t = kc + (i >> 6); col = c0 + (i & 63); }
            else { t = kc + (i & 31); col = c0 + (i >> 5); }
            const bool ok = col < g.n && t < K;
            gdbl *p = t >= K1 ? (gdbl *)g.B2 + ((long)col * ldb2 + (t - K1))
                              : (gdbl *)g.B + (g.btrans ? (long)t * ldb + col : (long)col * ldb + t);
            rbv[q] = *(ok ? p : zero);
        }
    };
    auto commit = [&]() {
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const int i = tid + 256 * q;
            As[(i >> 7) * BG_AP + (i & 127)] = ra[q];
        }
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const int i = tid + 256 * q;
            if (g.btrans) Bs[(i >> 6) * BG_BP + (i & 63)] = rbv[q];
            else Bs[(i & 31) * BG_BP + (i >> 5)] = rbv[q];
        }
    };
    const int lr = lane & 15, lk = lane >> 4, wr = wv * 32;
    d4h acc[2][4];
    for (int a = 0; a < 2; a++)
        for (int b = 0; b < 4; b++) acc[a][b] = (d4h){0.0, 0.0, 0.0, 0.0};
    stage(0);
    commit();
    __syncthreads();
    for (int kc = 0; kc < K; kc += BG_BK) {
        const bool more = kc + BG_BK < K;
        if (more) stage(kc + BG_BK);  // in flight while this chunk multiplies
        const int ksteps = min(BG_BK, ((K - kc) + 3) & ~3);
        for (int kq = 0; kq < ksteps; kq += 4) {
            const double *ap = As + (kq + lk) * BG_AP + wr + lr;
            const double *bp = Bs + (kq + lk) * BG_BP + lr;
            const double a0 = ap[0], a1 = ap[16];
            const double b0 = bp[0], b1 = bp[16], b2 = bp[32], b3 = bp[48];
            acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(b0, a0, acc[0][0], 0, 0, 0);
            acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(b1, a0, acc[0][1], 0, 0, 0);
            acc[0][2] = __builtin_amdgcn_mfma_f64_16x16x4f64(b2, a0, acc[0][2], 0, 0, 0);
            acc[0][3] = __builtin_amdgcn_mfma_f64_16x16x4f64(b3, a0, acc[0][3], 0, 0, 0);
            acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(b0, a1, acc[1][0], 0, 0, 0);
            acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(b1, a1, acc[1][1], 0, 0, 0);
            acc[1][2] = __builtin_amdgcn_mfma_f64_16x16x4f64(b2, a1, acc[1][2], 0, 0, 0);
            acc[1][3] = __builtin_amdgcn_mfma_f64_16x16x4f64(b3, a1, acc[1][3], 0, 0, 0);
        }
        __syncthreads();  // every wavefront is done with this chunk
        if (more) {
            commit();
            __syncthreads();
        }
    }
    // The B fragment is the MFMA's first operand, so that a lane's four results lie along a
    // row of C (columns lk, lk + 4, ...) and the 16 lanes of a store hold 16 adjacent
    // rows: each store writes 128-byte runs of C's columns, not 32-byte ones.  The
    // products and their order are the same.
    for (int b = 0; b < 4; b++)
        for (int i = 0; i < 4; i++) {
            const int col = c0 + b * 16 + lk + 4 * i;
            if (col >= g.n) continue;
            const long pc = g.cmap ? (long)((const __attribute__((address_space(1))) int *)g.cmap)[col] - g.cmoff : (long)col;
            gdblw *cp = (gdblw *)g.C + pc * g.ldc;
            for (int a = 0; a < 2; a++) {
                const int row = rb + wr + a * 16 + lr;
                if (row < g.nrow) cp[row] = g.beta ? (cp[row] + acc[a][b][i]) : acc[a][b][i];
            }
        }
}

// ---------------------------------------------------------------------------
// The same batched GEMM with wide tiles for large items: block = BM x BN outputs,
// wavefronts of (16 TA) x (16 TB) each (TA x TB accumulators of 16 x 16), k in chunks of
// BK staged through LDS (DB: two slabs, one barrier per chunk) with the next chunk in
// registers meanwhile.  nz > 0 numbers the blocks with the column block fastest
// (blockIdx.x = row block * nz + column block, blockIdx.z = 0), so the blocks of one row
// panel of A run together and the panel comes from HBM once; nz = 0 takes the row block
// from blockIdx.x and the column block from blockIdx.z.  Measured (FP64 MFMA peak 78.6
// TF/s):
//   * square products of order 8192: 256 x 128 with sixteen 32 x 64 wavefronts 52.7 TF/s,
//     eight 64 x 64 wavefronts 45.7, k_bgemm 34.8; below about 3000 rows and columns
//     there are too few blocks to fill the 256 CUs and k_bgemm is faster;
//   * the HSS multiply's steps at n = 32768: the tile follows the step's widest item
//     (128 x 64, 128 x 128 or 256 x 144), 24-38 % faster than k_bgemm.
// The k-steps of 4 run in the same order as in k_bgemm, so all give the same bits.
// ---------------------------------------------------------------------------
template <int BM, int BN, int BK, int DB, int TA, int TB>
__global__ __launch_bounds__((BM / (16 * TA)) * (BN / (16 * TB)) * 64) void k_bgemm_w(const BG *items, int nz)
{
    constexpr int WM = 16 * TA, WN = 16 * TB;  // rows and columns of one wavefront's tile
    constexpr int NT = (BM / WM) * (BN / WN) * 64;
    constexpr int AP = BM + 4, BP = BN + 4;
    // staged elements per thread; a slab that does not split evenly over the threads
    // (BN = 144) leaves the last round partly idle
    constexpr int QA = (BM * BK + NT - 1) / NT, QB = (BN * BK + NT - 1) / NT;
    constexpr bool EA = QA * NT == BM * BK, EB = QB * NT == BN * BK;
    __shared__ double Asb[(DB ? 2 : 1) * BK * AP];
    __shared__ double Bsb[(DB ? 2 : 1) * BK * BP];
    double *As = Asb, *Bs = Bsb;
    const BG g = items[blockIdx.y];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int bx = nz ? (int)blockIdx.x / nz : (int)blockIdx.x, bz = nz ? (int)blockIdx.x % nz : (int)blockIdx.z;
    const int rb = bx * BM, c0 = bz * BN;
    if (rb >= g.nrow || c0 >= g.n) return;  // the whole block
    const int K1 = g.k, K = g.k + g.k2;
    const long lda = g.lda, lda2 = g.lda2, ldb = g.ldb, ldb2 = g.ldb2;
    // staging: A element i = tid + NT q at (row rb + i % BM, k kc + i / BM); B element i at
    // (k kc + i / BN, column c0 + i % BN) for btrans, (k kc + i % BK, column c0 + i / BK)
    // column-major
    double ra[QA], rbv[QB];
    // Every staged element is one unconditional global load, an element outside the
    // operands reading a global zero, so no load sits in a branch and nothing uses the
    // loaded value before the commit (a branch around loads, or a select on their values,
    // makes the compiler wait for them at once, which serialises the prefetch with the
    // MFMAs).
    gdbl *const zero = (gdbl *)&bg_zero;
    auto stage = [&](int kc) {
#pragma unroll
        for (int q = 0; q < QA; q++) {
            const int i = tid + NT * q, row = rb + (i % BM), t = kc + i / BM;
            const bool ok = (EA || i < BM * BK) && row < g.nrow && t < K;
            gdbl *p = t < K1 ? (gdbl *)g.A + (row + (long)t * lda) : (gdbl *)g.A2 + (row + (long)(t - K1) * lda2);
            ra[q] = *(ok ? p : zero);
        }
#pragma unroll
        for (int q = 0; q < QB; q++) {
            const int i = tid + NT * q;
            int t, col;
            if (g.btrans) { t = kc + i / BN; col = c0 + i % BN; }
            else { t = kc + i % BK; col = c0 + i / BK; }
            const bool ok = (EB || i < BN * BK) && col < g.n && t < K;
            gdbl *p = t >= K1 ? (gdbl *)g.B2 + ((long)col * ldb2 + (t - K1))
                              : (gdbl *)g.B + (g.btrans ? (long)t * ldb + col : (long)col * ldb + t);
            rbv[q] = *(ok ? p : zero);
        }
    };
    auto commit = [&](double *Ad, double *Bd) {
#pragma unroll
        for (int q = 0; q < QA; q++) {
            const int i = tid + NT * q;
            if (EA || i < BM * BK) Ad[(i / BM) * AP + (i % BM)] = ra[q];
        }
#pragma unroll
        for (int q = 0; q < QB; q++) {
            const int i = tid + NT * q;
            if (!EB && i >= BN * BK) continue;
            if (g.btrans) Bd[(i / BN) * BP + (i % BN)] = rbv[q];
            else Bd[(i % BK) * BP + (i / BK)] = rbv[q];
        }
    };
    const int lr = lane & 15, lk = lane >> 4;
    const int wr = (wv % (BM / WM)) * WM, wc = (wv / (BM / WM)) * WN;
    d4h acc[TA][TB];
#pragma unroll
    for (int a = 0; a < TA; a++)
#pragma unroll
        for (int b = 0; b < TB; b++) acc[a][b] = (d4h){0.0, 0.0, 0.0, 0.0};
    stage(0);
    commit(As, Bs);
    __syncthreads();
    for (int kc = 0; kc < K; kc += BK) {
        const bool more = kc + BK < K;
        if (more) stage(kc + BK);  // in flight while this chunk multiplies
        const int ksteps = min(BK, ((K - kc) + 3) & ~3);
        for (int kq = 0; kq < ksteps; kq += 4) {
            const double *ap = As + (kq + lk) * AP + wr + lr;
            const double *bp = Bs + (kq + lk) * BP + wc + lr;
            double av[TA], bv[TB];
#pragma unroll
            for (int a = 0; a < TA; a++) av[a] = ap[16 * a];
#pragma unroll
            for (int b = 0; b < TB; b++) bv[b] = bp[16 * b];
#pragma unroll
            for (int a = 0; a < TA; a++)
#pragma unroll
                for (int b = 0; b < TB; b++)
                    acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[b], av[a], acc[a][b], 0, 0, 0);
        }
        if (DB) {
            // the other slab was last read before the previous barrier: fill it now, then
            // one barrier makes it readable and frees this one
            if (more) {
                double *An = (As == Asb) ? Asb + BK * AP : Asb, *Bn = (Bs == Bsb) ? Bsb + BK * BP : Bsb;
                commit(An, Bn);
                As = An;
                Bs = Bn;
            }
            __syncthreads();
        } else {
            __syncthreads();  // every wavefront is done with this chunk
            if (more) {
                commit(As, Bs);
                __syncthreads();
            }
        }
    }
    // first operand B, as in k_bgemm: 128-byte runs of C's columns per store
#pragma unroll
    for (int b = 0; b < TB; b++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int col = c0 + wc + b * 16 + lk + 4 * i;
            if (col >= g.n) continue;
            const long pc = g.cmap ? (long)((const __attribute__((address_space(1))) int *)g.cmap)[col] - g.cmoff : (long)col;
            gdblw *cp = (gdblw *)g.C + pc * g.ldc;
#pragma unroll
            for (int a = 0; a < TA; a++) {
                const int row = rb + wr + a * 16 + lr;
                if (row < g.nrow) cp[row] = g.beta ? (cp[row] + acc[a][b][i]) : acc[a][b][i];
            }
        }
}
template __global__ void k_bgemm_w<256, 128, 16, 1, 2, 4>(const BG *, int);
template __global__ void k_bgemm_w<128, 128, 16, 1, 2, 4>(const BG *, int);
template __global__ void k_bgemm_w<128, 64, 16, 1, 1, 4>(const BG *, int);
template __global__ void k_bgemm_w<128, 48, 16, 1, 1, 3>(const BG *, int);
template __global__ void k_bgemm_w<128, 32, 16, 1, 1, 2>(const BG *, int);
template __global__ void k_bgemm_w<128, 96, 16, 1, 2, 3>(const BG *, int);
template __global__ void k_bgemm_w<256, 144, 16, 1, 2, 9>(const BG *, int);

// X(:, t) = Q2(:, t): the K surviving old eigenvectors of each HSS merge packed
// densely (mdlaed2.f90:467-499), zero outside each column's support.
__global__ __launch_bounds__(WG) void k_gatherx(const Merge *mg, const int *hidx, const int *col_start, int nh,
                                                const Prob *probs, Work W, int cur, double *X, const long *xoff)
{
    int h = 0;
    {
        int lo = 0, hi = nh - 1, b = blockIdx.x;
        while (lo < hi) { int md = (lo + hi + 1) >> 1; if (col_start[md] <= b) lo = md; else hi = md - 1; }
        h = lo;
    }
    const Merge M = mg[hidx[h]];
    const int t = blockIdx.x - col_start[h];
    const Prob P = probs[M.prob];
    const int slot = W.vm[cur][M.s + W.indx[M.s + t] - 1];
    const int lo = W.supp_lo[slot], hi = W.supp_hi[slot];
    const double *src = P.q + (long)(slot - P.off) * P.ld - P.off;
    double *dst = X + xoff[h] + (long)t * M.n - M.s;
    for (int r = M.s + threadIdx.x; r < M.s + M.n; r += WG) dst[r] = (r >= lo && r < hi) ? src[r] : 0.0;
}

// dense C(i,j) = u_i v_j / (f_i - lambda_j) with accurate differences
// (CauchylikeEig with identity permutations), used when a merge's HSS form cannot
// be built within the LDS / arena limits
__global__ __launch_bounds__(WG) void k_cbuild(const HssMerge *hm, int h, double *C)
{
    const HssMerge H = hm[h];
    long KK = (long)H.K * H.K;
    for (long e = (long)blockIdx.x * WG + threadIdx.x; e < KK; e += (long)gridDim.x * WG) {
        int i = (int)(e % H.K) + 1, j = (int)(e / H.K) + 1;
        double den = (i <= j) ? (A1(H.FF, i) - A1(H.FF, j)) - A1(H.DIFL, j)
                              : (A1(H.FF, i) - A1(H.FF, j + 1)) - A1(H.DIFR, j);
        if (H.sq) den = den * (A1(H.FF, i) + A1(H.D0, j));
        C[e] = A1(H.U0, i) * A1(H.V0, j) / den;
    }
}

// 256 threads per node when a launch has nodes for every CU twice over, 512 when
// it has fewer (the upper tree levels): the search over the node's columns is the
// sequential part of every pivot step
template __global__ void k_hss_rowcomp<256, false>(const HssMerge *, const HssNode *, int, double, int);
template __global__ void k_hss_rowcomp<512, false>(const HssMerge *, const HssNode *, int, double, int);
template __global__ void k_hss_colcomp<256, false>(const HssMerge *, const HssNode *, int, double, int);
template __global__ void k_hss_colcomp<512, false>(const HssMerge *, const HssNode *, int, double, int);
template __global__ void k_hss_rowcomp<256, true>(const HssMerge *, const HssNode *, int, double, int);
template __global__ void k_hss_rowcomp<512, true>(const HssMerge *, const HssNode *, int, double, int);
template __global__ void k_hss_colcomp<256, true>(const HssMerge *, const HssNode *, int, double, int);
template __global__ void k_hss_colcomp<512, true>(const HssMerge *, const HssNode *, int, double, int);

// ===========================================================================
// General Cauchy-like matrices A(i,j) = u(i) v(j) / (d(i) - f(j)), direct
// differences: cauchy2hss (CauchyHss_VP2.f90:387-613).  The reference walks the
// tree in post order with a stack of compressed skeleton rows and columns, so a
// node's compression sees the skeletons of the nodes before it; that order fixes
// the ranks, and it is kept: one workgroup walks the tree, and every RRLU step
// (rrluCauchy, :7-134, rho = 1.02, a swap check every 10 steps) runs across the
// workgroup's threads, its scalar decisions taken identically by every thread from
// the same values.  Every element's operations and their order are the Fortran's.
//
// The bound is the latency of the pivot steps, one after another on one CU: both sides of
// a compression sit in LDS (up to C2H_LDS doubles; global scratch beyond), one instance of
// the step's code serves rows and columns of leaves and parents (eight inlined copies made
// 69 KB, more than the instruction cache), the next step's searches run inside the update
// pass, and W, needed only by the swap check and the generator, is formed ten steps at a
// time with a thread per entry.  n = 2000, leaf 64: 50.7 ms before, 17.2 now.
// ===========================================================================
#define C2H_NW (C2H_WG / 64)

// first largest |U(i) / (X(i) - y)| over i = k .. n (index i - k + 1), i from i0 by step
template <class DP>
__device__ __forceinline__ VI c2h_max(DP X, DP U, double y, int k, int n, int i0, int step)
{
    VI x = {0.0, 0};
    for (int i = k + i0; i <= n; i += step) x = vi_better(x, VI{fabs(A1(U, i) / (A1(X, i) - y)), i - k + 1});
    return x;
}

// rrluCauchy (:7-134) of the M x N matrix A(i) V(j) / (X(i) - Y(j)) with the pivoting of
// CauchyPivtG (:191-243) and CauchyPivtG_CP (:246-296); returns Rk.  U: the row generators
// of the Schur complement, W: those of the interpolation; T1, T2: M scratch each.
template <class DP, class IP>
__device__ __forceinline__ int c2h_rrlu(DP X, DP A, DP U, DP W, DP T1, DP T2, IP PL, DP Y, DP V, double tol, int M, int N,
                                     VI *red, int *s_ii, int *s_nsw)
{
    const int tid = threadIdx.x, lane = tid & 63, mn = M < N ? M : N;
    const double rho = 1.02;
    int tog = 0;
    for (int j = 1 + tid; j <= M; j += C2H_WG) { A1(U, j) = A1(A, j); A1(PL, j) = j; }
    __syncthreads();
    auto swapr = [&](int a, int b) {
        const double xa = A1(X, a), xb = A1(X, b), ua = A1(U, a), ub = A1(U, b), aa = A1(A, a), ab = A1(A, b);
        const int pa = A1(PL, a), pb = A1(PL, b);
        A1(X, a) = xb; A1(X, b) = xa;
        A1(U, a) = ub; A1(U, b) = ua;
        A1(A, a) = ab; A1(A, b) = aa;
        A1(PL, a) = pb; A1(PL, b) = pa;
    };
    auto swapc = [&](int a, int b) {
        const double ya = A1(Y, a), yb = A1(Y, b), va = A1(V, a), vb = A1(V, b);
        A1(Y, a) = yb; A1(Y, b) = ya;
        A1(V, a) = vb; A1(V, b) = va;
    };
    // W of steps 1 .. K from that of steps 1 .. k0: step q multiplies W(j), j < q, by
    // (Y(q) - X(j)) / (X(q) - X(j)) and sets W(q) = (X(q) - Y(q)) / A(q) times, then over,
    // (Y(j) - X(q)), (X(j) - X(q)) for j = 1 .. q - 1.  Positions 1 .. q of X, Y and A do not
    // change between step q and the next swap check, so ten steps' factors come at once.
    auto wsteps = [&](int k0, int K) {
        for (int j = 1 + tid; j <= K; j += C2H_WG) {
            const double xj = A1(X, j);
            double w;
            if (j > k0) {
                w = (xj - A1(Y, j)) / A1(A, j);
                for (int q = 1; q < j; q++) w = w * (A1(Y, q) - xj) / (A1(X, q) - xj);
            } else {
                w = A1(W, j);
            }
            for (int q = (j > k0 ? j : k0) + 1; q <= K; q++) w = w * ((A1(Y, q) - xj) / (A1(X, q) - xj));
            A1(W, j) = w;
        }
        __syncthreads();
    };
    int Rk = mn, kw = 0;  // kw: steps W holds
    double amax = 0.0;
    bool pre = false;     // pre_l, pre_u hold this step's first searches
    VI pre_l = {0.0, 0}, pre_u = {0.0, 0};
    for (int k = 1; k <= mn; k++) {
        VI L, R;
        if (pre) {
            L = pre_l;
            R = pre_u;
        } else {
            L = c2h_max(X, U, A1(Y, k), k, M, tid, C2H_WG);
            R = c2h_max(Y, V, A1(X, k), k, N, tid, C2H_WG);
            block_argmax2_t<C2H_NW>(L, R, red, tog);
        }
        const double junkL = L.v * fabs(A1(V, k)), junkU = R.v * fabs(A1(U, k));
        const double piv = fabs(A1(U, k) * A1(V, k) / (A1(X, k) - A1(Y, k)));
        if (!(junkL <= piv && junkU <= piv)) {
            int flg = (junkL > junkU) ? 1 : 0, jjL = L.i, jjU = R.i;
            // a row swap is made after the column search it feeds and its barrier; a column
            // swap first waits until every thread has read position k
            if (flg == 0) __syncthreads();
            // every round moves a strictly larger entry into the pivot, so finite data ends
            // within M + N rounds; the bound only guarantees an exit for overflowed generators
            for (int round = 0; round < M + N + 2; round++) {
                if (flg == 1) {
                    const int jr = jjL + k - 1;
                    jjU = block_argmax_t<C2H_NW>(c2h_max(Y, V, A1(X, jr), k, N, tid, C2H_WG), red, tog).i;
                    if (tid == 0) swapr(k, jr);
                    if (jjU == 1) break;
                }
                if (tid == 0) swapc(k, jjU + k - 1);
                __syncthreads();
                // a few hundred rows: every wavefront searches them by itself
                if (M - k < 256) jjL = wave_argmax<64>(c2h_max(X, U, A1(Y, k), k, M, lane, 64)).i;
                else jjL = block_argmax_t<C2H_NW>(c2h_max(X, U, A1(Y, k), k, M, tid, C2H_WG), red, tog).i;
                if (jjL == 1) break;
                flg = 1;
            }
            __syncthreads();
        }
        double ukk = A1(U, k) * A1(V, k) / (A1(X, k) - A1(Y, k));
        amax = fmax(amax, fabs(ukk));
        if (fabs(ukk) < tol * amax) {
            // complete pivoting over the Schur complement
            VI best = {0.0, 0};
            int bestrow = 1;
            for (int j = k + tid; j <= N; j += C2H_WG) {
                const double yj = A1(Y, j);
                double mv = 0.0;
                int mi = 0;
                for (int i = k; i <= M; i++) {
                    const double u = A1(U, i), den = A1(X, i) - yj;
                    if (mi != 0 && !may_exceed(u, den, mv)) continue;
                    const double x = fabs(u / den);
                    if (mi == 0 || x > mv) { mv = x; mi = i - k + 1; }
                }
                const VI c = {fabs(mv * A1(V, j)), j - k + 1};
                const VI nb = vi_better(best, c);
                if (nb.i == c.i) bestrow = mi;
                best = nb;
            }
            const VI win = block_argmax_t<C2H_NW>(best, red, tog);
            if (best.i == win.i && win.i > 0) *s_ii = bestrow;
            __syncthreads();
            if (tid == 0) {
                swapr(k, *s_ii + k - 1);
                swapc(k, win.i + k - 1);
            }
            __syncthreads();
            ukk = A1(U, k) * A1(V, k) / (A1(X, k) - A1(Y, k));
            amax = fmax(amax, fabs(ukk));
            if (fabs(ukk) < tol * amax) { Rk = k - 1; break; }
        }
        // generators of the next Schur complement; unless a swap check follows, the next
        // step's first searches run inside the passes
        const double Xk = A1(X, k), Yk = A1(Y, k);
        const bool fuse = k + 1 <= mn && k % 10 != 0;
        const double Xn = fuse ? A1(X, k + 1) : 0.0, Yn = fuse ? A1(Y, k + 1) : 0.0;
        VI x1 = {0.0, 0}, y1 = {0.0, 0};
        for (int j = k + 1 + tid; j <= M; j += C2H_WG) {
            const double xj = A1(X, j), u = A1(U, j) * (xj - Xk) / (xj - Yk);
            A1(U, j) = u;
            if (fuse) x1 = vi_better(x1, VI{fabs(u / (xj - Yn)), j - k});
        }
        for (int j = k + 1 + tid; j <= N; j += 2 * C2H_WG) {
            const int j2 = j + C2H_WG;
            const double ya = A1(Y, j), va = A1(V, j), yb = A1(Y, min(j2, N)), vb = A1(V, min(j2, N));
            const double na = va * (ya - Yk) / (ya - Xk), nb = vb * (yb - Yk) / (yb - Xk);
            A1(V, j) = na;
            if (j2 <= N) A1(V, j2) = nb;
            if (fuse) {
                y1 = vi_better(y1, VI{fabs(na / (ya - Xn)), j - k});
                if (j2 <= N) y1 = vi_better(y1, VI{fabs(nb / (yb - Xn)), j2 - k});
            }
        }
        pre = fuse;
        if (fuse) {
            block_argmax2_t<C2H_NW>(x1, y1, red, tog);
            pre_l = x1;
            pre_u = y1;
        } else {
            __syncthreads();
        }
        if (k % 10 != 0) continue;
        wsteps(kw, k);
        kw = k;
        // each swap raises |det| of the pivot block by more than rho; bounded all the same
        for (int sw = 0; sw < 2 * M + 8; sw++) {
            // searchMax2 (:137-163): the largest entry of Mat_N(i, j) = U(k+i) W(j) / (X(k+i) - X(j)),
            // G lanes to a column
            VI x = {0.0, 0};
            int xrow = 1;
            const int G = scan_lanes(k, C2H_WG), g = tid & (G - 1);
            for (int jc = 1 + tid / G; jc - tid / G <= k; jc += C2H_WG / G) {
                VI e = {0.0, 0};
                if (jc <= k) {
                    const double xj = A1(X, jc);
                    for (int i = 1 + g; i <= M - k; i += G)
                        e = vi_better(e, VI{fabs(A1(U, k + i) / (A1(X, k + i) - xj)), i});
                }
                e = group_argmax(e, G);
                if (jc <= k) {
                    const VI c = {e.v * fabs(A1(W, jc)), jc};
                    const VI nb = vi_better(x, c);
                    if (nb.i == c.i) xrow = e.i > 0 ? e.i : 1;
                    x = nb;
                }
            }
            const VI win = block_argmax_t<C2H_NW>(x, red, tog);
            if (!(win.v > rho)) break;
            if (x.i == win.i && g == 0) *s_ii = xrow;
            __syncthreads();
            const int ii = win.i, jj = *s_ii + k;
            const double Dii = A1(X, ii), Djj = A1(X, jj);
            for (int j = k + 1 + tid; j <= N; j += C2H_WG) A1(V, j) = A1(V, j) * ((A1(Y, j) - Dii) / (A1(Y, j) - Djj));
            for (int j = k + 1 + tid; j <= M; j += C2H_WG)
                if (j != jj) A1(U, j) = A1(U, j) * ((A1(X, j) - Djj) / (A1(X, j) - Dii));
            for (int j = 1 + tid; j <= k; j += C2H_WG) {
                const double xj = A1(X, j), yj = A1(Y, j);
                if (j != ii) A1(W, j) = A1(W, j) * ((xj - Dii) / (xj - Djj));
                // the factors of U(jj) and W(ii); 1 at j = ii leaves the products' bits
                A1(T1, j) = j == ii ? 1.0 : (Dii - xj) / (Dii - yj);
                A1(T2, j) = j == ii ? 1.0 : (yj - Djj) / (xj - Djj);
            }
            __syncthreads();
            if (tid == 0) {
                const double yii = A1(Y, ii);
                double uj = A1(A, ii) * ((Dii - Djj) / (Dii - yii));
                double wi = (Djj - yii) / A1(A, jj);
                for (int j = 1; j <= k; j++) {
                    uj = uj * A1(T1, j);
                    wi = wi * A1(T2, j);
                }
                const double xi = A1(X, ii), xj = A1(X, jj), ai = A1(A, ii), aj = A1(A, jj);
                const int pi = A1(PL, ii), pj = A1(PL, jj);
                A1(U, jj) = uj;
                A1(W, ii) = wi;
                A1(PL, ii) = pj; A1(PL, jj) = pi;
                A1(X, ii) = xj; A1(X, jj) = xi;
                A1(A, ii) = aj; A1(A, jj) = ai;
                *s_nsw += 1;
            }
            __syncthreads();
        }
    }
    wsteps(kw, Rk);
    return Rk;
}

// comprcauchy (:616-725) of one side of node `nodi` ('r': M node rows against N outside
// columns, 'c': M node columns against N outside rows): gathers the node's side from
// (A, Au) at m0 and the outside from (B, Bv) -- the stacked skeletons 1 .. cs - 1, then the
// originals after `last` --, runs the RRLU, writes the interpolative generator
// (Cauchylike2, :743-778, in the node's order) to the arena and the skeleton back to
// (A, Au) at o0.  The six node arrays lie st apart at w.  Returns its rank, -1 when the arena is full.
template <class DP, class IP>
__device__ __forceinline__ int c2h_compr(const C2H &C, bool row, DP w, long st, IP PL, IP inv, DP Y, DP V, int m0, int M, int cs,
                                         int last, int N, int o0, int nodi, long &top, VI *red, int *s_ii, int *s_nsw)
{
    const int tid = threadIdx.x;
    DP X = w, A = w + st, U = w + 2 * st, W = w + 3 * st, T1 = w + 4 * st, T2 = w + 5 * st;
    double *Ag = row ? C.D : C.F, *Aug = row ? C.U : C.V, *Bg = row ? C.F : C.D, *Bvg = row ? C.V : C.U;
    for (int j = tid; j < M; j += C2H_WG) { X[j] = A1(Ag, m0 + j); A[j] = A1(Aug, m0 + j); W[j] = 0.0; }
    for (int j = tid; j < N; j += C2H_WG) {
        const int src = (j < cs - 1) ? j + 1 : last + 1 + (j - (cs - 1));
        Y[j] = A1(Bg, src);
        V[j] = A1(Bvg, src);
    }
    __syncthreads();
    const int Rk = c2h_rrlu<DP, IP>(X, A, U, W, T1, T2, PL, Y, V, C.tol, M, N, red, s_ii, s_nsw);
    // inverse of the row permutation
    for (int i = 1 + tid; i <= M; i += C2H_WG) A1(inv, A1(PL, i)) = i;
    const int r = Rk < M ? Rk : M;
    const long off = top;
    __syncthreads();
    if (off + (long)M * r > C.arena_cap) {
        if (tid == 0) atomicOr(C.err, 2);
        return -1;
    }
    double *Q = C.arena + off;
    for (long e = tid; e < (long)M * r; e += C2H_WG) {
        // rows: Q is M x r, entry (i, j); columns: r x M, entry (i, j) of the transpose
        const int a = (int)(e % (row ? M : r)) + 1, b = (int)(e / (row ? M : r)) + 1;
        const int i = row ? a : b, j = row ? b : a, s = A1(inv, i);
        double q;
        if (Rk >= M || s <= r) q = (s == j) ? 1.0 : 0.0;
        else q = A1(U, s) * A1(W, j) / (A1(X, s) - A1(X, j));
        Q[e] = q;
    }
    if (tid == 0) {
        if (row) { C.usz[2 * (nodi - 1)] = M; C.usz[2 * (nodi - 1) + 1] = r; C.pu[nodi - 1] = off; }
        else { C.vsz[2 * (nodi - 1)] = r; C.vsz[2 * (nodi - 1) + 1] = M; C.pv[nodi - 1] = off; }
    }
    top = off + (long)M * r;
    for (int j = tid; j < Rk; j += C2H_WG) { A1(Ag, o0 + j) = X[j]; A1(Aug, o0 + j) = A[j]; }
    __syncthreads();
    return Rk;
}

// Cauchylike (Cauchylike.f90:1-13) into a (lda), M x N
__device__ void g_cfill(double *a, int lda, const double *D, const double *F, const double *u, const double *v, int M,
                        int N)
{
    for (long e = threadIdx.x; e < (long)M * N; e += C2H_WG) {
        const int i = (int)(e % M) + 1, j = (int)(e / M) + 1;
        a[(i - 1) + (long)(j - 1) * lda] = A1(u, i) * A1(v, j) / (A1(D, i) - A1(F, j));
    }
}

__global__ __launch_bounds__(C2H_WG) void k_cauchy2hss(C2H C, int lds_cap)
{
    extern __shared__ double hss_dyn[];  // lds_cap doubles
    __shared__ VI red[4 * C2H_NW];
    __shared__ int s_ii, s_nsw;
    typedef __attribute__((address_space(3))) int lint;
    const int tid = threadIdx.x, lda = C.n;
    long top = 0;               // arena bump, the same in every thread
    int ns = 1;
    int *lsr = C.lsr, *lsc = C.lsc;
    if (tid == 0) { A1(lsr, 1) = 1; A1(lsc, 1) = 1; s_nsw = 0; }
    __syncthreads();
    for (int i = 1; i <= C.ltr; i++) {
        const int c1 = C.ch[2 * (i - 1)], c2 = C.ch[2 * (i - 1) + 1];
        const int l1 = C.rng[2 * (i - 1)], l2 = C.rng[2 * (i - 1) + 1];
        const bool leaf = c1 == 0;
        if (leaf) {
            const int mi = l2 - l1 + 1;
            g_cfill(C.dd + C.pd[i - 1], mi, C.D + l1 - 1, C.F + l1 - 1, C.U + l1 - 1, C.V + l1 - 1, mi, mi);
            if (tid == 0) C.dsz[i - 1] = mi;
        } else {  // parent: B of both children, then its own compressions
            for (int t = 0; t < 2; t++) {
                const int cr = t ? ns - 1 : ns - 2, cc = t ? ns - 2 : ns - 1, cnode = t ? c2 : c1;
                const int r0 = A1(lsr, cr), mi = A1(lsr, cr + 1) - r0, q0 = A1(lsc, cc), ni = A1(lsc, cc + 1) - q0;
                if (top + (long)mi * ni > C.arena_cap) { if (tid == 0) atomicOr(C.err, 2); return; }
                g_cfill(C.arena + top, mi, C.D + r0 - 1, C.F + q0 - 1, C.U + r0 - 1, C.V + q0 - 1, mi, ni);
                if (tid == 0) { C.bsz[2 * (cnode - 1)] = mi; C.bsz[2 * (cnode - 1) + 1] = ni; C.pb[cnode - 1] = top; }
                top += (long)mi * ni;
            }
            if (i == C.ltr) break;
        }
        __syncthreads();
        // a leaf's rows and columns are the originals l1 .. l2, a parent's the merged
        // skeletons of its children; the skeletons of the nodes before it and the
        // originals after it are outside
        const int base = leaf ? ns : ns - 2;  // stack position this node's skeletons go to
        for (int side = 0; side < 2; side++) {
            const bool row = side == 0;
            const int *own = row ? lsr : lsc, *oth = row ? lsc : lsr;
            const int m0 = leaf ? l1 : A1(own, base), M = leaf ? l2 - l1 + 1 : A1(own, ns) - A1(own, base);
            const int cs = base == 1 ? 1 : A1(oth, base), N = lda - l2 + cs - 1, o0 = A1(own, base);
            __syncthreads();  // every thread has read the stack before it changes
            int Rk;
            if (7L * M + 2L * N + 2 <= lds_cap) {
                ldbl *w = (ldbl *)hss_dyn;
                Rk = c2h_compr<ldbl *, lint *>(C, row, w, (long)M, (lint *)(w + 6 * M), (lint *)(w + 6 * M) + M, w + 7 * M,
                                               w + 7 * M + N, m0, M, cs, l2, N, o0, i, top, red, &s_ii, &s_nsw);
            } else {
                Rk = c2h_compr<gdblw *, gint *>(C, row, (gdblw *)C.S, (long)C.n, (gint *)C.PL, (gint *)C.PU, (gdblw *)C.Fi,
                                                (gdblw *)C.Vi, m0, M, cs, l2, N, o0, i, top, red, &s_ii, &s_nsw);
            }
            if (Rk < 0) return;
            if (tid == 0) A1(row ? lsr : lsc, base + 1) = o0 + Rk;
            __syncthreads();
        }
        ns = base + 1;
    }
    if (tid == 0) *C.nswap = (unsigned long long)s_nsw;
}

// the dense general Cauchy-like matrix (fallback for a tree of one leaf)
__global__ __launch_bounds__(WG) void k_cfill_general(int n, const double *d, const double *f, const double *u,
                                                      const double *v, double *a)
{
    for (long e = blockIdx.x * (long)WG + threadIdx.x; e < (long)n * n; e += (long)gridDim.x * WG) {
        const int i = (int)(e % n), j = (int)(e / n);
        a[e] = u[i] * v[j] / (d[i] - f[j]);
    }
}
