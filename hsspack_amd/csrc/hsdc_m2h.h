// Dense-to-HSS construction: descriptors and launch limits shared by its kernels
// (hsdc_mat2hss.hip) and the host that plans them (hsdc_api.hip).
#pragma once
#include <algorithm>

// One node's compression problem of one side: T (w x m, column-major, ld w) gathered
// from C; the result basis (m x m, ld m, columns in descending singular value order),
// its singular values and rank.  side 0: block row (basis U), 1: block column (W).
struct M2hJob {
    int rs, rn, cs, cn;  // the node's rows and columns in C
    int w, m;            // context length and own length of this side
    long toff;           // T, then R (m x m), V (m x m) at toff + w m, + m m
    long boff;           // basis (m x m) and singular values (m)
    int lq;              // 1: a second QR before the Jacobi sweeps; 0: the sketch of a sampled side
};

// New rows or columns of C: block a is formed from a job pair's basis, or is an old block.
struct M2hBlk {
    int start, count;  // new block in C' (rows or columns)
    int src;           // >= 0: job pair (2 src = row side, 2 src + 1 = column side); < 0: -1 - old block
    int ostart, ocount;  // the old rows / columns it is formed from
};

// Copies of one level's generators into the arena: kind 0 U (m x r from the row basis),
// 1 V = W^T (r x m from the column basis), 2 B (a block of C'), 3 D (a block of A).
struct M2hCopy {
    int kind, rows, cols, job;  // job: the basis (kinds 0, 1)
    int r0, c0;                 // the block's origin in its source (kinds 2, 3)
    long dst;                   // arena / leaf-block offset
};

// One chunk of rows of a tall matrix (rows x m at src, ld lds) and the place of its R (m x m
// at dst, ld ldd).
struct M2hChunk {
    long src, dst;
    int rows, m, lds, ldd;
};

#define M2H_SVD_WG 1024  // threads per block of k_m2h_svd and k_m2h_qr
#define M2H_LDS 19800    // LDS doubles they may take (160 KB less their static arrays)
#define M2H_QM 100       // columns of a QR in LDS: R and V both fit up to 99
#define M2H_QR_ROWS 512  // rows of a QR in LDS: eight registers of a wavefront hold a column
#define M2H_QR_COLS 96   // columns that the tree of QRs takes: a chunk has 2 m rows or more
static_assert(2 * M2H_QM * M2H_QM > M2H_LDS && M2H_QM <= 128, "R and V in LDS: fewer than M2H_QM columns");
static_assert(M2H_QR_COLS <= M2H_QM && M2H_LDS / M2H_QR_COLS >= 2 * M2H_QR_COLS && M2H_QR_ROWS >= 2 * M2H_QR_COLS,
              "every stage of the tree shrinks the matrix");
static_assert(8 * (M2H_LDS + 3 * M2H_QM + M2H_SVD_WG / 64) + 64 <= 160 * 1024, "LDS of a workgroup");

// rows of an m-column matrix that one workgroup reduces in LDS (0: more columns than the
// tree reduction takes)
inline int m2h_qr_rows(int m) { return m < 1 || m > M2H_QR_COLS ? 0 : std::min(M2H_QR_ROWS, M2H_LDS / m); }

__global__ void k_m2h_gather(const M2hJob *jobs, const double *C, long ldc, double *S);
__global__ void k_m2h_svd(const M2hJob *jobs, double *S, double *Bs, double tol, int *rank, int *err, int lds_cap);
__global__ void k_m2h_qr(const M2hChunk *ch, double *S);
__global__ void k_m2h_sketch(const M2hJob *jobs, const M2hJob *sk, const double *S0, double *S,
                             unsigned long long seed);
__global__ void k_m2h_rows(const M2hBlk *blk, int nb, const M2hJob *jobs, const double *Bs, const double *C, long ldc,
                           int nc, double *out, long ldo);
__global__ void k_m2h_cols(const M2hBlk *blk, int nb, const M2hJob *jobs, const double *Bs, const double *Tr, long ldt,
                           int nnc, double *out);
__global__ void k_m2h_copy(const M2hCopy *cp, const M2hJob *jobs, const double *Bs, const double *Cn, long ldcn,
                           const double *A, long lda, double *arena, double *dd);
