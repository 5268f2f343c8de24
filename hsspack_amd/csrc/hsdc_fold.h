// Ordered folds over the poles of a merge: for every root a product or a sum of one
// term per pole, taken in pole order (the order fixes the bits), each term costing one
// or two FP64 divides.
//
// A thread per root spends the chain's length in divides and leaves most of the chip
// idle (K / 64 wavefronts per merge): 55 us for the product of K = 1000 roots, 67 ns per
// pole and level at K = 32768.  The divides do not depend on each other, only the
// fold does, so a block of nine wavefronts splits the two: eight form the terms of a
// chunk of OF_P poles for R roots (lane = root, 64 / R poles per wavefront at a time)
// into one half of a double buffer while the ninth folds the previous chunk in order
// and stages the pole values of the next chunks.  One barrier per chunk.  Measured,
// before and after: K = 1000 product 55 -> 16 us, column norms 81 -> 14 us; K = 32768
// 1.8 -> 1.18 ms and 2.4 -> 1.14 ms (of 0.75 ms that the divides alone take at 90 cycles a
// wavefront); K = 1400 dense vectors 182 -> 18 us.  Chunks of 32 poles (three blocks per
// CU instead of two): 1.45 ms at K = 32768.
#pragma once
#include <algorithm>
#include "hsdc_internal.h"

#define OF_P 64    // poles per chunk
#define OF_WG 576  // eight wavefronts that form terms, one that folds them

template <int NV>
struct FoldLds {
    double ring[4][NV][OF_P];  // pole values of four chunks
    double buf[2][OF_P * 64];  // terms of two chunks, R per pole
};

// How a level's nch chunks of 256 roots are split over blocks: `parts` blocks to a chunk,
// each taking the chunk's roots R at a time from its own part.  Blocks of 16 roots are
// four times as many, and a chunk of poles costs them the folding wavefront's steps instead
// of the divides: the faster split as long as every one of them has a CU to itself, 16
// chunks on 256 CUs.  From 17 on two would share a CU, and 64 roots, which keep all eight
// wavefronts' lanes on divides, are faster.  One merge of K roots (secular equation, product
// and norms), 16 against 64 roots, us: K = 2040 151 / 175, 4000 338 / 389, 4090 344 / 399,
// 4500 529 / 486, 6000 717 / 657, 12000 2040 / 1658, 16384 3660 / 2710, 25000 8516 / 6250,
// 32500 13124 / 9300.
// From 1024 chunks on (many small merges) a block takes whole chunks: finding a part's
// merge costs two dependent loads, more than the work of a part that is empty (2048
// chunks of K = 40: 112 us against 422 for the vector build; 800 chunks of K = 500: 420
// against 480 the other way round).
#define OF_NARROW 16  // chunks up to which a block takes 16 roots
struct FoldSplit { int R, parts; };
__device__ __forceinline__ FoldSplit fold_split(int nch)
{
    return nch >= 1024 ? FoldSplit{64, 1} : nch > OF_NARROW ? FoldSplit{64, 4} : FoldSplit{16, 16};
}
// Blocks to launch for at most nch chunks of 256 roots (the kernels stride): enough for the
// narrow split too, which fewer chunks than the bound may take
inline int fold_grid(long nch)
{
    const long b = nch >= 1024 ? nch : nch > OF_NARROW ? std::max(4 * nch, 16L * OF_NARROW) : 16 * nch;
    return (int)(b < 1 ? 1 : b > 2048 ? 2048 : b);
}

// The fold of poles [0, n) for the R roots of this block: on the ninth wavefront's
// lanes < R the result, starting from acc.  F gives
//   raw(p)           first loads of pole p (a value type)
//   vals(raw, v)     the NV values staged for it (dependent loads go here)
//   term<W>(v, p)    the term of pole p for this thread's root, values v[q * OF_P];
//                    W = 1: p lies below every root of the block, 2: above, 0: either or
//                    the root's own pole
//   fold(acc, t)     the fold
// Every thread of the block calls it; n is uniform.  A block barrier precedes the
// return, so the LDS may be reused at once.
// r0: the block's first root (0-based).  n >= 1.
template <int R, int NV, class F>
__device__ __forceinline__ double ordered_fold(const F &f, int n, int r0, double acc, FoldLds<NV> &S)
{
    constexpr int Q = 64 / R, U = OF_P / (8 * Q);  // poles per wavefront step, steps per chunk
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, sl = lane & (OF_P - 1);
    const int nch = (n + OF_P - 1) / OF_P;
    const bool folder = wv == 8;
    decltype(f.raw(0)) nx{};
    if (folder) {
        // chunks 0 and 1 staged, chunk 2's first loads under way
        for (int c = 0; c < 2; c++) {
            double v[NV];
            f.vals(f.raw(min(c * OF_P + sl, n - 1)), v);
#pragma unroll
            for (int q = 0; q < NV; q++) S.ring[c][q][sl] = v[q];
        }
        nx = f.raw(min(2 * OF_P + sl, n - 1));
    }
    __syncthreads();
    for (int c = 0; c <= nch; c++) {
        if (!folder) {
            if (c < nch) {
                // a wavefront's poles are adjacent, so that its broadcast reads pair up
                const double *v = &S.ring[c & 3][0][0] + wv * U * Q + lane / R;
                double *b = S.buf[c & 1] + wv * U * 64 + lane;
                const int p = c * OF_P + wv * U * Q + lane / R;
                double t[U];
                if ((c + 1) * OF_P <= r0) {
#pragma unroll
                    for (int u = 0; u < U; u++) t[u] = f.template term<1>(v + u * Q, p + u * Q);
                } else if (c * OF_P >= r0 + R) {
#pragma unroll
                    for (int u = 0; u < U; u++) t[u] = f.template term<2>(v + u * Q, p + u * Q);
                } else {
#pragma unroll
                    for (int u = 0; u < U; u++) t[u] = f.template term<0>(v + u * Q, p + u * Q);
                }
#pragma unroll
                for (int u = 0; u < U; u++) b[u * 64] = t[u];
            }
        } else {
            double v[NV];
            if (c + 2 < nch) f.vals(nx, v);
            if (c > 0 && lane < R) {
                const double *b = S.buf[(c - 1) & 1] + lane;
                const int cn = min(OF_P, n - (c - 1) * OF_P);
                int p = 0;
                for (; p + 16 <= cn; p += 16) {
                    double t[16];
#pragma unroll
                    for (int u = 0; u < 16; u++) t[u] = b[(p + u) * R];
#pragma unroll
                    for (int u = 0; u < 16; u++) acc = f.fold(acc, t[u]);
                }
                for (; p < cn; p++) acc = f.fold(acc, b[p * R]);
            }
            if (c + 2 < nch) {
#pragma unroll
                for (int q = 0; q < NV; q++) S.ring[(c + 2) & 3][q][sl] = v[q];
                nx = f.raw(min((c + 3) * OF_P + sl, n - 1));
            }
        }
        __syncthreads();
    }
    return acc;
}
