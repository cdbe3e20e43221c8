// lu2mi_lu.hip -- GPU-resident blocked recursive LU with partial pivoting and
// the solve that follows it, in lu2's factor form.
//
// Algorithm (lu2.c:1122-1144 lumcolumn, lu2.c:1088-1120 recursive panel,
// lu2.c:524-581 process_right_part, lu2.c:485-521 solve_triangle,
// lu2.c:110-116 backward_sub) re-planned for one MI355X:
//
//  per nb-block i:
//    panel(i, nb)                       recursive halving down to a W-column leaf
//      leaf   : one persistent kernel factors W columns of rows [c, n) held in
//               registers; one exchange per column brings every workgroup
//               the pivot candidates of all (wavefront argmax, lowest row on
//               ties) together with the candidate rows, so the winning row
//               arrives with the decision.  It also forms the leaf's W x W
//               block of (D^-1 L11)^-1.
//      rowperm: the leaf's swaps applied to the other panel columns, with
//               the 1/d scaling of the L part left of the diagonal
//               (lu2.c:1112-1118, lu2tlib.c:1119-1126).
//      node   : right half rows scaled by 1/d, TRSM by the explicit inverse
//               (lu2.c:467-512) as an MFMA GEMM, trailing MFMA GEMM
//               (lu2.c:580), and the off-diagonal block of the inverse.
//    rowperm of the block's nb swaps over columns [i+nb, n] (b included),
//      1/d scaling, block rows redirected to the staging buffer (awork)
//    U12 = Linv * staging                 (lu2.c:511-512)
//    A22 -= L21 * U12                     (lu2.c:580, 97.7% of the flops)
//  back substitution on the unit-upper U (lu2.c:110-116), blocked.
//
//  Lookahead schedule (default): the block-level steps run first on the next
//  panel's nb columns only, panel(i+nb) then starts on a second stream, and
//  the block's remaining columns follow on the first; same arithmetic per
//  element as the serial order.  Optionally, up to 256 columns of a panel
//  run as one persistent launch (subpanel_kernel) with grid barriers between
//  the steps above.
//
// Layout in HBM: lu2's row-major augmented matrix, lda >= n+1 (RDIM = n+16
// in lu2.c:28), b in column n.  Row-major rows are contiguous, so row swaps
// and scalings are coalesced along rows.
#include "lu2mi_internal.h"
#include "lu2mi_dev.h"
#include "lu2mi_gemm_tile.h"
#include "lu2mi_leaf.h"
#include <stdarg.h>
#include <stdlib.h>
#include <string.h>
#include <chrono>
#include <vector>

// drand48 on the device: jump-ahead generator in lu2mi_dev.h.
using namespace lu2mi_rng;

__global__ __launch_bounds__(256) void randomsetmat_kernel(double *A, long lda, int n,
                                                           unsigned long long x0)
{
    const long r = blockIdx.x;
    const int t = threadIdx.x;
    // element (r, col) is draw number r*(n+1)+col; its value is the state
    // after draw+1 steps
    const unsigned long long first = (unsigned long long)r * (unsigned long long)(n + 1) + t + 1;
    const Lcg jump = lcg_pow(first);
    unsigned long long x = (jump.a * x0 + jump.c) & M48;
    const Lcg step = lcg_pow(256);
    double *row = A + r * lda;
    for (int col = t; col <= n; col += 256) {
        row[col] = (double)x * (1.0 / 281474976710656.0) - 0.5;
        x = (step.a * x + step.c) & M48;
    }
    for (long col = n + 1 + t; col < lda; col += 256) row[col] = 0.0;
}

// a[i][i] += sum_j |a[i][j]| over the n columns of A (diagonal dominance for
// the 16-bit solves); one workgroup per row, fixed reduction order
__global__ __launch_bounds__(256) void diag_dominant_kernel(double *A, long lda, int n)
{
    __shared__ double red[4];
    const long r = blockIdx.x;
    const int t = threadIdx.x;
    const double *row = A + r * lda;
    double s = 0.0;
    for (int c = t; c < n; c += 256) s += fabs(row[c]);
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((t & 63) == 0) red[t >> 6] = s;
    __syncthreads();
    if (t == 0) A[r * lda + r] += (red[0] + red[1]) + (red[2] + red[3]);
}

// maximum that keeps a NaN (fmax drops it): a NaN solution must not pass as
// a small residual
__device__ __forceinline__ double nan_max(double a, double b) { return (a > b || a != a) ? a : b; }

template <typename T>
__global__ __launch_bounds__(256) void rowperm_kernel(PermArgs<T> a)
{
    extern __shared__ unsigned char smem_raw[];
    __builtin_amdgcn_s_setprio(3);
    rowperm_strip<T>(a, blockIdx.x, (T *)smem_raw);
}

// The block-level permutation (lu2.c:524-556), pairs (i+k, orig[i+k]) and
// (piv[i+k], orig[piv[i+k]]), without LDS staging, in two
// launches over (pair, 1024-column chunk).  Destinations inside the block go
// to the staging buffer W (scaled by 1/d), so pass 0 reads A and writes only
// W.  A row below the block only ever receives content that started in the
// block (content that enters the block from below stays there), so pass 1
// reads block rows of A, which no pass writes, and writes rows below, which
// pass 1 never reads.  Every read of a row below happens in pass 0.
// first: the pairs are formed here from the block's pivots and origins (a
// launch of its own before), and kept for the remaining columns.
template <typename T>
__global__ __launch_bounds__(256) void staged_perm_kernel(PermArgs<T> a, int pass, const int *piv, const int *orig,
                                                          int *dst, int *src)
{
    const int pr = blockIdx.y;
    int d, sr;
    if (piv) {
        const int nb = a.w1 - a.w0;
        d = pr < nb ? a.w0 + pr : piv[a.w0 + pr - nb];
        sr = orig[d];
        if (blockIdx.x == 0 && pass == 0 && threadIdx.x == 0) {
            dst[pr] = d;
            src[pr] = sr;
        }
    } else {
        d = a.dst[pr];
        sr = a.src[pr];
    }
    const bool to_w = (d >= a.w0 && d < a.w1);
    if (to_w != (pass == 0)) return;
    const T *srow = a.A + (long)sr * a.lda;
    const bool scale = (d >= a.d0 && d < a.d1);
    const T sc = scale ? a.invd[d] : T(1);
    T *drow = to_w ? a.W + (long)(d - a.w0) * a.ldw - a.c0 : a.A + (long)d * a.lda;
    const int col0 = a.c0 + blockIdx.x * 1024;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int col = col0 + q * 256 + threadIdx.x;
        if (col < a.c1) {
            T v = srow[col];
            if (scale && col < a.sce) v *= sc;
            drow[col] = v;
        }
    }
}

// W[r][col] = A[r0+r][c0+col] * invd[r0+r]  (rows scaled by 1/d before the TRSM)
template <typename T>
__global__ void scale_copy_kernel(const T *A, long lda, int r0, int c0, int h, int nc, const T *invd,
                                  T *W)
{
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < (long)h * nc) {
        const int r = (int)(e / nc), col = (int)(e % nc);
        W[e] = A[(long)(r0 + r) * lda + c0 + col] * invd[r0 + r];
    }
}

// ---------------------------------------------------------------------------
// Recursion nodes of half-width h <= 64: one workgroup (one 64x64 tile) per
// step, and the steps that follow one another in the recursion -- the inverse
// blocks of the nodes that end at a leaf, deepest first, then the TRSM of the
// node whose left half they close -- in one launch.  Same arithmetic as the
// separate steps; what a launch costs is not its work (a step of its own 4-6
// us, of which 1-2 us arithmetic; together, alone on the device, 3.5 us for
// one TRSM to 29 us for three inverse blocks and a TRSM, 10.4 us on average)
// but being one more in the panel's chain.
//   inverse block: X21 = -inv22 * (L21 * inv11), tmp passes between the
//     products through memory
//   TRSM: X = inv(D^-1 L11) * (rows [c, c+h) of the right half scaled by 1/d),
//     the scaling done as the rows are loaded (the staging copy's values); the
//     tile reads all of its rows before it writes them back
struct NodeSteps {
    int ninv;               // inverse blocks, at most one per half-width 16, 32, 64
    int inv_c[3], inv_h[3];
    int trsm_c, trsm_h;     // trsm_h = 0: none
};
template <typename T>
__global__ __launch_bounds__(256) void node_steps64_kernel(T *A, long lda, NodeSteps ns, T *linv, int ldl, int i,
                                                           T *tmp, const T *invd)
{
    using namespace lu2mi_gemm;
    __shared__ Tile64Smem<T> sm;
    __builtin_amdgcn_s_setprio(3);
    auto fence = [&]() __attribute__((always_inline)) {
        __threadfence();
        __syncthreads();
    };
    GemmDesc g;
    for (int q = 0; q < ns.ninv; q++) {
        const int c = ns.inv_c[q], h = ns.inv_h[q];
        const long off = c - i;
        g.M = h; g.N = h; g.K = h; g.alpha = 1.0; g.beta = 0.0;
        g.lda = lda; g.ldb = ldl; g.ldc = h; g.a_lower = 0;
        gemm_tile64<T, true, EPI_SET>(g, A + (long)(c + h) * lda + c, linv + off * ldl + off, tmp, 0, 0, h, sm);
        fence();
        g.alpha = -1.0; g.lda = ldl; g.ldb = h; g.ldc = ldl; g.a_lower = 1;
        gemm_tile64<T, true, EPI_GENERAL>(g, linv + (off + h) * ldl + off + h, tmp, linv + (off + h) * ldl + off, 0,
                                          0, h, sm);
        fence();
    }
    if (ns.trsm_h) {
        const int c = ns.trsm_c, h = ns.trsm_h;
        const long off = c - i;
        g.M = h; g.N = h; g.K = h; g.alpha = 1.0; g.beta = 0.0;
        g.lda = ldl; g.ldb = lda; g.ldc = lda; g.a_lower = 1;
        T *X = A + (long)c * lda + c + h;
        gemm_tile64<T, true, EPI_SET>(g, linv + off * ldl + off, X, X, 0, 0, h, sm, invd + c);
    }
}
// column-major panel (m columns of ld rows, rows [r0, r0+R)) <-> row-major (R x ldp)
__global__ void cm_to_rm_kernel(const double *cm, long ld, int r0, int R, int m, double *rm, long ldp, int back)
{
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (long)R * m) return;
    const int r = (int)(e / m), col = (int)(e % m);
    if (back) ((double *)cm)[(long)col * ld + r0 + r] = rm[(long)r * ldp + col];
    else rm[(long)r * ldp + col] = cm[(long)col * ld + r0 + r];
}

template <typename T>
__global__ void fill_kernel(T *p, long count, T v)
{
    for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < count; e += (long)gridDim.x * blockDim.x)
        p[e] = v;
}

template <typename T>
__global__ void copy_col_kernel(const T *A, long lda, int n, int col, T *x)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < n) x[r] = A[(long)r * lda + col];
}

// ---------------------------------------------------------------------------
// Back substitution on the unit-upper U (lu2.c:110-116) in one persistent
// launch.  Rows are cut into 64-row blocks, solved bottom-up; block number
// idx (0 = bottom) belongs to workgroup idx % G (all G co-resident).  A
// workgroup accumulates U[block rows][solved block] * x[solved block] for
// every block below it as soon as the shared frontier (count of solved
// blocks) shows it solved -- the A tile of the next block it will need is
// loaded into registers before it waits -- then solves its 64x64 diagonal
// block right-looking in one wavefront (each finished x broadcast with
// readlane), publishes x with device-scope stores and advances the frontier.
// With 64-row blocks the adjacent block (the last one solved before this one)
// is left to wavefront 0: the other blocks' sums are reduced across lanes
// while that block is still being solved, its 64x64 tile waits transposed in
// LDS, and at the hand-over one wavefront applies it (lane = row) and goes on
// to the diagonal solve with no workgroup barrier in between.  x holds y on
// entry.  TF is the factor's element type, TX the vector's (FP64 for
// refinement).
constexpr int BSB = 64;

template <typename TF, typename TX, int BS>
__global__ __launch_bounds__(BS * 4) void backsub_kernel(const TF *__restrict__ A, long lda, int n, TX *x,
                                                         unsigned long long *front, int *err, int strict)
{
    // BS-row blocks, BS/16 waves of 16 rows each; the columns of a solved
    // block are taken 64 at a time (lane = column), in BS/64 halves
    constexpr int NT = BS * 4, NH = BS / 64;
    constexpr bool ADJ = (BS == 64);   // the adjacent block applied by wavefront 0
    __shared__ TF Ud[BS][BS + 1];
    __shared__ TF UaT[ADJ ? BS : 1][BS + 1];   // UaT[k][row]: the tile against the adjacent block
    __shared__ TX part[BS];
    __shared__ int s_front;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int nblk = (n + BS - 1) / BS;
    const int G = gridDim.x;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(x, 0, (int)(sizeof(TX) * n), 0x00020000);
    for (int idx = blockIdx.x; idx < nblk; idx += G) {
        const int b = nblk - 1 - idx;
        const int r0 = b * BS, r1 = min(n, r0 + BS), nrb = r1 - r0;
        for (int e = t; e < BS * BS; e += NT) {
            const int rr = e / BS, kk = e % BS;
            Ud[rr][kk] = (rr < nrb && kk < nrb) ? A[(long)(r0 + rr) * lda + r0 + kk] : TF(0);
        }
        if constexpr (ADJ) {
            // columns [r0 + BS, r0 + 2 BS) of the block's rows (none for the bottom block)
            const int c0 = r0 + BS, nc = min(BS, n - c0);
            for (int e = t; e < BS * BS; e += NT) {
                const int rr = e / BS, kk = e % BS;
                UaT[kk][rr] = (rr < nrb && kk < nc) ? A[(long)(r0 + rr) * lda + c0 + kk] : TF(0);
            }
        }
        // wave w accumulates rows r0 + 16w .. r0 + 16w + 15, lane = column in the solved block
        TX acc[16];
        TF pa[NH][16];
#pragma unroll
        for (int i = 0; i < 16; i++) acc[i] = TX(0);
        // the 64 columns h of solved block d for this thread: rows r0 + 16w + i,
        // column c0(d) + 64 h + lane
        auto fetch = [&](int d, int h, TF *v) {
            const int col = (nblk - 1 - d) * BS + 64 * h + lane;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int r = r0 + w * 16 + i;
                v[i] = (r < r1 && col < n) ? A[(long)r * lda + col] : TF(0);
            }
        };
        auto accumulate = [&](int d, int h, const TF *v) {
            const int col = (nblk - 1 - d) * BS + 64 * h + lane;
            const TX xv = (col < n) ? ld_buf(xr, (int)(sizeof(TX) * col), TX(0)) : TX(0);
#pragma unroll
            for (int i = 0; i < 16; i++) acc[i] += (TX)v[i] * xv;
        };
        // this block's y, loaded before the waits: only this workgroup writes
        // these rows of x, and only once it solves the block
        TX yv[NH];
        if (t < 64)
#pragma unroll
            for (int h = 0; h < NH; h++) yv[h] = (t + 64 * h < nrb) ? x[r0 + t + 64 * h] : TX(0);
        // solved blocks summed by all waves (lane = column): all below this
        // one, or all but the adjacent one
        const int need = ADJ ? idx - 1 : idx;
        int done = 0;
        if (need > 0)
#pragma unroll
            for (int h = 0; h < NH; h++) fetch(0, h, pa[h]);
        while (done < need) {
            if (t == 0) {
                unsigned long spins = 0;
                int f;
                while ((f = (int)ld_relaxed(front)) <= done) {
                    __builtin_amdgcn_s_sleep(1);
                    if (((++spins) & 1023) == 0) {
                        if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) { f = idx; break; }
                        if (spins > (1UL << 25)) {
                            __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            f = idx;
                            break;
                        }
                    }
                }
                s_front = f;
            }
            __syncthreads();
            const int F = min(s_front, need);
            acquire_seq(strict);
#pragma unroll
            for (int h = 0; h < NH; h++) accumulate(done, h, pa[h]);   // the prefetched tile
            int d = done + 1;
            if (NH == 1) {
                for (; d + 1 < F; d += 2) {      // blocks already solved: two tiles in flight
                    TF v0[16], v1[16];
                    fetch(d, 0, v0);
                    fetch(d + 1, 0, v1);
                    accumulate(d, 0, v0);
                    accumulate(d + 1, 0, v1);
                }
            }
            for (; d < F; d++) {
                TF v0[16], v1[16];
                fetch(d, 0, v0);
                if (NH > 1) fetch(d, NH - 1, v1);
                accumulate(d, 0, v0);
                if (NH > 1) accumulate(d, NH - 1, v1);
            }
            done = F;
            if (done < need)
#pragma unroll
                for (int h = 0; h < NH; h++) fetch(done, h, pa[h]);   // ahead of the next wait
            __syncthreads();
        }
#pragma unroll
        for (int i = 0; i < 16; i++) {
            TX v = acc[i];
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
            if (lane == 0) part[w * 16 + i] = v;
        }
        __syncthreads();
        if (t < 64) {
            // right-looking: x[rr] is final when step rr begins; rows above
            // subtract U[row][rr] x[rr]; lane t holds rows t + 64 h
            TX xt[NH];
#pragma unroll
            for (int h = 0; h < NH; h++) xt[h] = (t + 64 * h < nrb) ? yv[h] - part[t + 64 * h] : TX(0);
            if constexpr (ADJ) {
                if (idx > 0) {
                    // the adjacent block: this wavefront alone waits for it
                    unsigned long spins = 0;
                    while ((int)ld_relaxed(front) < idx) {
                        __builtin_amdgcn_s_sleep(1);
                        if (((++spins) & 1023) == 0) {
                            if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
                            if (spins > (1UL << 25)) {
                                if (lane == 0) __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                                break;
                            }
                        }
                    }
                    acquire_seq(strict);
                    const int ca = r0 + BS + lane;
                    const TX xa = (ca < n) ? ld_buf(xr, (int)(sizeof(TX) * ca), TX(0)) : TX(0);
                    TX s0 = TX(0), s1 = TX(0);
#pragma unroll
                    for (int k = 0; k < BS; k += 2) {
                        s0 += (TX)UaT[k][lane] * lane_bcast(xa, k);
                        s1 += (TX)UaT[k + 1][lane] * lane_bcast(xa, k + 1);
                    }
                    xt[0] -= s0 + s1;
                }
            }
            for (int rr = nrb - 1; rr > 0; rr--) {
                TX xk;
                if (NH == 1 || rr < 64) xk = lane_bcast(xt[0], rr & 63);
                else xk = lane_bcast(xt[NH - 1], rr & 63);
#pragma unroll
                for (int h = 0; h < NH; h++)
                    if (t + 64 * h < rr) xt[h] -= (TX)Ud[t + 64 * h][rr] * xk;
            }
#pragma unroll
            for (int h = 0; h < NH; h++)
                if (t + 64 * h < nrb) st_dev(x + r0 + t + 64 * h, xt[h]);
            // the block's x all come from this one wave, whose s_waitcnt
            // vmcnt(0) in publish_seq covers every lane's store
            if (!strict && t == 0) publish_seq(front, (unsigned long long)(idx + 1), 0);
        }
        __syncthreads();
        // strict: the workgroup barrier orders the other lanes' stores before
        // thread 0's release store
        if (strict && t == 0) publish_seq(front, (unsigned long long)(idx + 1), 1);
    }
}

// ---------------------------------------------------------------------------
// FP64 residual: per row |(A x)_i - b_i| and sum_j |a_ij|; per column sum |a_ij|.
// A wavefront takes RESID_ROWS rows, so each x[c] it loads serves all of them;
// each row is summed in the same order as by a wavefront of its own.
constexpr int RESID_ROWS = 4;
__global__ __launch_bounds__(256) void resid_rows_kernel(const double *A, long lda, int n, const double *x,
                                                         double *rerr, double *rabs)
{
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const long r0 = ((long)blockIdx.x * 4 + wave) * RESID_ROWS;
    if (r0 >= n) return;
    const int nr = (int)min((long)RESID_ROWS, (long)n - r0);
    const double *a = A + r0 * lda;
    double s[RESID_ROWS], sa[RESID_ROWS];
#pragma unroll
    for (int q = 0; q < RESID_ROWS; q++) s[q] = sa[q] = 0.0;
    // four columns' loads in flight per lane and row
#pragma unroll 4
    for (int c = lane; c < n; c += 64) {
        const double xc = x[c];
#pragma unroll
        for (int q = 0; q < RESID_ROWS; q++) {
            if (q < nr) {
                const double e = a[q * lda + c];
                s[q] = fma(e, xc, s[q]);
                sa[q] += fabs(e);
            }
        }
    }
#pragma unroll
    for (int q = 0; q < RESID_ROWS; q++) {
        for (int off = 32; off > 0; off >>= 1) {
            s[q] += __shfl_xor(s[q], off);
            sa[q] += __shfl_xor(sa[q], off);
        }
    }
    if (lane == 0) {
        for (int q = 0; q < nr; q++) {
            rerr[r0 + q] = fabs(s[q] - a[q * lda + n]);
            rabs[r0 + q] = sa[q];
        }
    }
}

// A workgroup takes 64 columns; its 16 waves take the rows r = w (mod 16), eight
// loads in flight each, and the 16 partial sums per column are added in a
// fixed order, so the result does not depend on timing.  HBM bound once enough
// loads are in flight: n = 20001 has 313 such column blocks, little more than
// one per CU, and with 4 waves of 4 loads the whole check took 1608 us,
// now 1522 with 696 for this kernel (the same sums in the same order).
constexpr int RESID_CW = 16;
__global__ __launch_bounds__(64 * RESID_CW) void resid_cols_kernel(const double *A, long lda, int n, double *cabs)
{
    __shared__ double part[RESID_CW][64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int col = blockIdx.x * 64 + lane;
    double s = 0.0;
    if (col < n) {
        const double *a = A + col;
#pragma unroll 8
        for (long r = wave; r < n; r += RESID_CW) s += fabs(a[r * lda]);
    }
    part[wave][lane] = s;
    __syncthreads();
    if (wave == 0 && col < n) {
        double p[4];
#pragma unroll
        for (int w = 0; w < 4; w++) p[w] = (part[w][lane] + part[w + 4][lane]) + (part[w + 8][lane] + part[w + 12][lane]);
        cabs[col] = (p[0] + p[1]) + (p[2] + p[3]);
    }
}

// out[0]=max rerr, [1]=max rabs, [2]=max cabs, [3]=max|x|, [4]=sum|x|, [5]=max|b|
__global__ __launch_bounds__(256) void resid_final_kernel(const double *A, long lda, int n, const double *x,
                                                          const double *rerr, const double *rabs,
                                                          const double *cabs, double *out)
{
    __shared__ double sh[6][256];
    const int t = threadIdx.x;
    double v[6] = {0, 0, 0, 0, 0, 0};
    // one workgroup, a chain of loads: eight steps' loads in flight (the
    // column b alone is a cache line per row)
#pragma unroll 8
    for (int r = t; r < n; r += 256) {
        v[0] = nan_max(v[0], rerr[r]);
        v[1] = nan_max(v[1], rabs[r]);
        v[2] = nan_max(v[2], cabs[r]);
        v[3] = nan_max(v[3], fabs(x[r]));
        v[4] += fabs(x[r]);
        v[5] = nan_max(v[5], fabs(A[(long)r * lda + n]));
    }
    for (int k = 0; k < 6; k++) sh[k][t] = v[k];
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if (t < st)
            for (int k = 0; k < 6; k++) sh[k][t] = (k == 4) ? sh[k][t] + sh[k][t + st] : nan_max(sh[k][t], sh[k][t + st]);
        __syncthreads();
    }
    if (t < 6) out[t] = sh[t][0];
    if (t == 0) {
        // the scaled forms: HPL-2 with eps = 2^-53, and lu2_mpi.c:2170-2229's
        // resid1..3 with lu2's eps = 2e-16
        const double eps = 1.1102230246251565e-16, eps_lu2 = 2e-16, dn = (double)n;
        const double r = sh[0][0], ainf = sh[1][0], a1 = sh[2][0], xinf = sh[3][0], x1 = sh[4][0], bmax = sh[5][0];
        out[6] = r / (eps * (ainf * xinf + bmax) * dn);
        out[7] = r / (eps_lu2 * a1 * dn);
        out[8] = r / (eps_lu2 * a1 * x1);
        out[9] = r / (eps_lu2 * ainf * xinf * dn);
    }
}

// Scratch of the residual entry point that allocates nothing
// (lu2mi_residual_dev_noalloc): per-row |(Ax)_i - b_i| and sum_j |a_ij|, per
// column sum_i |a_ij| -- 3n doubles for n up to LU2MI_RESID_NMAX.  Each
// device holds its own copy until the process ends; host code reaches it only
// through the address lu2mi_scratch_address() obtains (ctx->d_scratch), and
// calls that overlap on one device share it (they race).
static __device__ __align__(256) double scratch[3 * (size_t)LU2MI_RESID_NMAX];

// ===========================================================================
// host side
// ===========================================================================
static char g_errmsg[512];
void lu2mi_set_error_msg(const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_errmsg, sizeof g_errmsg, fmt, ap);
    va_end(ap);
}
extern "C" const char *lu2mi_last_error(void) { return g_errmsg; }

int lu2mi_dev_buf(void **p, size_t *cur, size_t need)
{
    if (*cur >= need && *p) return LU2MI_OK;
    if (*p) (void)hipFree(*p);
    *p = nullptr;
    *cur = 0;
    if (need == 0) return LU2MI_OK;
    if (hipMalloc(p, need) != hipSuccess) {
        *p = nullptr;
        lu2mi_set_error_msg("hipMalloc(%zu) failed", need);
        return LU2MI_ERR_NOMEM;
    }
    *cur = need;
    return LU2MI_OK;
}

int lu2mi_ctx_reserve(lu2mi_ctx *ctx, int n, int nb, int esz)
{
    (void)esz;
    if (n <= ctx->n_cap && nb <= ctx->nb_cap && ctx->d_w) return LU2MI_OK;
    const int ncap = n > ctx->n_cap ? n : ctx->n_cap;
    const int nbcap = nb > ctx->nb_cap ? nb : ctx->nb_cap;
    (void)hipFree(ctx->d_piv); (void)hipFree(ctx->d_orig); (void)hipFree(ctx->d_invd);
    (void)hipFree(ctx->d_invd_f); (void)hipFree(ctx->d_pairs); (void)hipFree(ctx->d_linv);
    (void)hipFree(ctx->d_tmp); (void)hipFree(ctx->d_y);
    ctx->d_piv = nullptr; ctx->d_orig = nullptr; ctx->d_invd = nullptr; ctx->d_invd_f = nullptr;
    ctx->d_pairs = nullptr; ctx->d_linv = nullptr; ctx->d_tmp = nullptr; ctx->d_y = nullptr;
    LU2MI_CHECK(hipMalloc(&ctx->d_piv, sizeof(int) * (size_t)ncap));
    LU2MI_CHECK(hipMalloc(&ctx->d_orig, sizeof(int) * (size_t)ncap));
    LU2MI_CHECK(hipMalloc(&ctx->d_invd, sizeof(double) * (size_t)ncap));
    LU2MI_CHECK(hipMalloc(&ctx->d_invd_f, sizeof(float) * (size_t)ncap));
    // pairs and Linv: two of each (blocks i and i+1 alternate, so the next
    // panel can be factored while block i's rows are still being moved);
    // d_tmp: the panel's h x h product scratch, then its h x h staging rows
    LU2MI_CHECK(hipMalloc(&ctx->d_pairs, sizeof(int) * 2 * 4 * (size_t)(nbcap > 64 ? nbcap : 64)));
    LU2MI_CHECK(hipMalloc(&ctx->d_linv, sizeof(double) * 2 * (size_t)nbcap * nbcap));
    LU2MI_CHECK(hipMalloc(&ctx->d_tmp, sizeof(double) * 2 * (size_t)nbcap * nbcap));
    LU2MI_CHECK(hipMalloc(&ctx->d_y, sizeof(double) * 4 * (size_t)ncap + 64));
    size_t wneed = sizeof(double) * (size_t)nbcap * (size_t)(ncap + 1);
    LU2MI_TRY(lu2mi_dev_buf(&ctx->d_w, &ctx->w_bytes, wneed));
    // leaf exchange slots, then the sub-panel grid barrier word (both cleared
    // at the start of every factorization)
    size_t sneed = SLOTS_BYTES + 256;
    LU2MI_TRY(lu2mi_dev_buf(&ctx->d_slots, &ctx->slots_bytes, sneed));
    ctx->n_cap = ncap;
    ctx->nb_cap = nbcap;
    return LU2MI_OK;
}

// ---------------------------------------------------------------------------
template <typename T> struct Prec;
template <> struct Prec<double> {
    static int gemm(const GemmDesc &g, hipStream_t s) { return lu2mi_gemm_f64(g, s); }
    static double *invd(lu2mi_ctx *c) { return c->d_invd; }
};
template <> struct Prec<float> {
    static int gemm(const GemmDesc &g, hipStream_t s) { return lu2mi_gemm_f32(g, s); }
    static float *invd(lu2mi_ctx *c) { return c->d_invd_f; }
};

template <typename T>
static int gemm_call(lu2mi_ctx *ctx, int M, int N, int K, double alpha, const T *A, long lda,
                     const T *B, long ldb, double beta, T *C, long ldc, int a_lower, int tag = 0)
{
    GemmDesc g;
    g.M = M; g.N = N; g.K = K; g.batch = 1;
    g.alpha = alpha; g.beta = beta;
    g.A = A; g.lda = lda; g.sA = 0;
    g.B = B; g.ldb = ldb; g.sB = 0;
    g.C = C; g.ldc = ldc; g.sC = 0;
    g.a_lower = a_lower;
    g.tag = tag;
    return Prec<T>::gemm(g, ctx->stream);
}

// x <- U^-1 x with the unit-upper U stored in A (one persistent launch)
template <typename TF, typename TX, int BS>
static int backsub_bs(lu2mi_ctx *ctx, const TF *A, long lda, int n, TX *x)
{
    const int nblk = (n + BS - 1) / BS;
    int per_cu = 0;
    LU2MI_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)backsub_kernel<TF, TX, BS>, 4 * BS, 0));
    // every workgroup the device keeps co-resident: more workgroups mean
    // shorter backlogs of solved tiles each
    int G = per_cu * ctx->num_cu < nblk ? per_cu * ctx->num_cu : nblk;
    if (G < 1) G = 1;
    LU2MI_CHECK(hipMemsetAsync(ctx->d_bar, 0, sizeof(unsigned long long), ctx->stream));
    hipLaunchKernelGGL((backsub_kernel<TF, TX, BS>), dim3(G), dim3(4 * BS), 0, ctx->stream, A, lda, n, x, ctx->d_bar,
                       ctx->d_err, ctx->strict_sync);
    LU2MI_CHECK(hipGetLastError());
    return LU2MI_OK;
}

// 64-row blocks, or 128 (LU2MI_OPT_BACKSUB128): half as many frontier steps,
// each a cross-workgroup hand-over, for a longer diagonal solve per step
template <typename TF, typename TX>
static int backsub(lu2mi_ctx *ctx, const TF *A, long lda, int n, TX *x)
{
    if (ctx->backsub128) return backsub_bs<TF, TX, 128>(ctx, A, lda, n, x);
    return backsub_bs<TF, TX, BSB>(ctx, A, lda, n, x);
}

template <typename T>
struct Factor {
    lu2mi_ctx *ctx;
    T *A;
    long lda;
    int n, nb, compat, W;
    T *linv, *tmp, *wbuf;
    T *pwbuf;              // the panel's staging rows (wbuf holds the block's)
    int *pairs;
    T *linv_base = nullptr;   // two nb x nb inverses, alternating by block
    int *pairs_base = nullptr;
    // when set, every block keeps its inverse diagonal block and its row
    // pairs here (for later solves with the stored factors)
    T *linv_all = nullptr;
    int *pairs_all = nullptr;

    int leaf(int i, int c)
    {
        const int R = n - c;
        // rows per thread: at most 64 workgroups for the 16-wide leaf (fewer
        // slots to gather per column), 128 for the 32-wide one
        const int gcap = (W == 16) ? 64 : 128;
        int rpt = (R + NTL * gcap - 1) / (NTL * gcap);
        if (rpt < 1) rpt = 1;
        if (W == 32 && rpt > 2) rpt = 2;
        if (W == 16 && rpt > 4) rpt = 4;
        if (rpt == 3) rpt = 4;
        // up to 512 rows in one workgroup: no exchange through memory (above
        // that four rows per thread would cost more: 1000 rows 47 us, and with
        // the exchange 4096 rows take 43.5 us at one row per thread)
        if (R <= 2 * NTL) rpt = (R <= NTL) ? 1 : 2;
        const int G = (R + NTL * rpt - 1) / (NTL * rpt);
        if (G > LEAF_GMAX) {
            lu2mi_set_error_msg("leaf: %d rows need %d workgroups (> %d)", R, G, LEAF_GMAX);
            return LU2MI_ERR_UNSUPPORTED;
        }
        LeafArgs<T> la;
        la.A = A; la.lda = lda; la.n = n; la.c = c; la.i = i; la.compat = compat; la.G = G;
        la.piv = ctx->d_piv; la.orig = ctx->d_orig; la.invd = Prec<T>::invd(ctx);
        la.pair_dst = pairs; la.pair_src = pairs + 2 * W;
        la.linv = linv; la.ldl = nb;
        la.slots = (unsigned long long *)ctx->d_slots;
        la.seq_base = ctx->bar_count; la.err = ctx->d_err;
        void *args[] = {&la};
        const void *fn = nullptr;
        if (W == 32) fn = (rpt == 1) ? (const void *)leaf_kernel<T, 32, 1> : (const void *)leaf_kernel<T, 32, 2>;
        else fn = (rpt == 1) ? (const void *)leaf_kernel<T, 16, 1>
                 : (rpt == 2) ? (const void *)leaf_kernel<T, 16, 2> : (const void *)leaf_kernel<T, 16, 4>;
        // All G workgroups must be resident together (each waits for the
        // messages of all, once per column).  An ordinary launch on an
        // otherwise idle device places them all when occupancy allows it; the
        // runtime's cooperative launch is not used because it holds a
        // per-device resource that a second process on the same GPU cannot
        // get.  The wait's bounded spin turns any shortfall into
        // LU2MI_ERR_DEVICE rather than a hang.
        int per_cu = 0;
        LU2MI_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, NTL, 0));
        if ((long)per_cu * ctx->num_cu < G) {
            lu2mi_set_error_msg("leaf: %d workgroups cannot be co-resident (%d per CU x %d CUs)", G, per_cu,
                                ctx->num_cu);
            return LU2MI_ERR_UNSUPPORTED;
        }
        LU2MI_CHECK(hipLaunchKernel(fn, dim3(G), dim3(NTL), args, 0, ctx->stream));
        ctx->bar_count += (unsigned long long)W;
        // apply the leaf's swaps to the other panel columns; L part (columns
        // left of the leaf) of the leaf's diagonal rows scaled by 1/d
        return rowperm(pairs, pairs + 2 * W, 2 * W, i, i + nb, c, c + W, c, c, c + W, nullptr, 0, 0, 0);
    }

    int rowperm(const int *dst, const int *src, int np, int c0, int c1, int k0, int k1, int sce, int d0,
                int d1, T *Wb, long ldw, int w0, int w1, bool first = false)
    {
        if (c1 <= c0) return LU2MI_OK;
        static bool lds_attr = false;
        if (!lds_attr) {
            LU2MI_CHECK(hipFuncSetAttribute((const void *)rowperm_kernel<T>,
                                            hipFuncAttributeMaxDynamicSharedMemorySize, 131072));
            lds_attr = true;
        }
        PermArgs<T> p;
        p.A = A; p.lda = lda; p.dst = dst; p.src = src; p.np = np;
        p.c0 = c0; p.c1 = c1; p.k0 = k0; p.k1 = k1; p.sce = sce; p.d0 = d0; p.d1 = d1;
        p.invd = Prec<T>::invd(ctx); p.W = Wb; p.ldw = ldw; p.w0 = w0; p.w1 = w1;
        if (Wb && w0 == d0 && w1 == d1 && k0 == k1) {
            // block level: destinations in [w0, w1) are the block's rows
            p.sw = 0;
            const dim3 grid((c1 - c0 + 1023) / 1024, np);
            for (int pass = 0; pass < 2; pass++)
                hipLaunchKernelGGL(staged_perm_kernel<T>, grid, dim3(256), 0, ctx->stream, p, pass,
                                   first ? (const int *)ctx->d_piv : nullptr, (const int *)ctx->d_orig, (int *)dst,
                                   (int *)src);
            LU2MI_CHECK(hipGetLastError());
            return LU2MI_OK;
        }
        // strip width: every source row of the strip fits in LDS; strips of at
        // least 64 bytes per row, and narrow enough for ~2 strips per CU
        const int seg = 64 / (int)sizeof(T);
        int sw = (c1 - c0 + 2 * ctx->num_cu - 1) / (2 * ctx->num_cu);
        sw = (sw + seg - 1) / seg * seg;
        if (sw > 128) sw = 128;
        const int swmax = (int)(131072 / (np * (int)sizeof(T)));
        if (sw > swmax) sw = swmax;
        if (sw < 1) {
            lu2mi_set_error_msg("rowperm: %d row pairs do not fit in LDS", np);
            return LU2MI_ERR_UNSUPPORTED;
        }
        p.sw = sw;
        const int strips = (c1 - c0 + sw - 1) / sw;
        const size_t shm = (size_t)np * sw * sizeof(T);
        hipLaunchKernelGGL(rowperm_kernel<T>, dim3(strips), dim3(256), shm, ctx->stream, p);
        LU2MI_CHECK(hipGetLastError());
        return LU2MI_OK;
    }

    // rows per thread and workgroups of a 16-wide leaf over R rows: at most
    // 64 workgroups (fewer slots to gather per column), up to 4 rows each
    static void leaf16_shape(int R, int &rpt, int &G)
    {
        rpt = (R + NTL * 64 - 1) / (NTL * 64);
        if (rpt < 1) rpt = 1;
        if (rpt > 4) rpt = 4;
        if (rpt == 3) rpt = 4;
        G = (R + NTL * rpt - 1) / (NTL * rpt);
    }

    // the sub-panel kernel applies to 16-wide leaves on 16-byte aligned rows
    bool sub_ok(int w) const
    {
        constexpr long EPV = 16 / sizeof(T);
        auto al = [](const void *p) { return ((uintptr_t)p & 15) == 0; };
        return ctx->sub_w > 0 && W == SUB_W && w <= ctx->sub_w && w <= SUB_WMAX && w >= W && al(A) &&
               lda % EPV == 0 && nb % EPV == 0 && al(linv) && al(pwbuf) && al(tmp);
    }

    int subpanel(int i, int c, int w)
    {
        int rpt, G;
        leaf16_shape(n - c, rpt, G);
        if (G > LEAF_GMAX) {
            lu2mi_set_error_msg("sub-panel: %d rows need %d workgroups (> %d)", n - c, G, LEAF_GMAX);
            return LU2MI_ERR_UNSUPPORTED;
        }
        SubArgs<T> sa;
        LeafArgs<T> &la = sa.leaf;
        la.A = A; la.lda = lda; la.n = n; la.c = c; la.i = i; la.compat = compat; la.G = G;
        la.piv = ctx->d_piv; la.orig = ctx->d_orig; la.invd = Prec<T>::invd(ctx);
        la.pair_dst = pairs; la.pair_src = pairs + 2 * SUB_W;
        la.linv = linv; la.ldl = nb;
        la.slots = (unsigned long long *)ctx->d_slots;
        la.seq_base = ctx->bar_count; la.err = ctx->d_err;
        sa.nb = nb; sa.w = w;
        // strips of at least 64 bytes per row, about one per workgroup
        const int seg = 64 / (int)sizeof(T);
        int sw = (nb + G - 1) / G;
        sw = (sw + seg - 1) / seg * seg;
        sa.sw = sw > SUB_SWMAX ? SUB_SWMAX : sw;
        sa.wbuf = pwbuf; sa.tmp = tmp;
        sa.gbar = (unsigned long long *)((char *)ctx->d_slots + SLOTS_BYTES);
        sa.gbar_base = ctx->gbar_count;
        const void *fn = (rpt == 1) ? (const void *)subpanel_kernel<T, 1>
                         : (rpt == 2) ? (const void *)subpanel_kernel<T, 2> : (const void *)subpanel_kernel<T, 4>;
        // all G workgroups must be co-resident (grid barriers), as for the leaf
        int per_cu = 0;
        LU2MI_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, NTL, 0));
        if ((long)per_cu * ctx->num_cu < G) {
            lu2mi_set_error_msg("sub-panel: %d workgroups cannot be co-resident (%d per CU x %d CUs)", G, per_cu,
                                ctx->num_cu);
            return LU2MI_ERR_UNSUPPORTED;
        }
        void *args[] = {&sa};
        LU2MI_CHECK(hipLaunchKernel(fn, dim3(G), dim3(NTL), args, 0, ctx->stream));
        ctx->bar_count += (unsigned long long)w;   // W sequence numbers per leaf
        ctx->gbar_count += (unsigned long long)G * sub_barriers(w / SUB_W);
        return LU2MI_OK;
    }

    NodeSteps steps{};   // inverse blocks due, not launched yet

    // the inverse blocks due, and the TRSM of node (c, 2h) if h > 0
    int node_steps(int i, int c, int h)
    {
        steps.trsm_c = c;
        steps.trsm_h = h;
        if (steps.ninv || h) {
            hipLaunchKernelGGL(node_steps64_kernel<T>, dim3(1), dim3(256), 0, ctx->stream, A, lda, steps, linv, nb, i,
                               tmp, Prec<T>::invd(ctx));
            LU2MI_CHECK(hipGetLastError());
        }
        steps = NodeSteps{};
        return LU2MI_OK;
    }

    int panel(int i, int c, int w)
    {
        if (sub_ok(w)) return subpanel(i, c, w);
        if (w <= W) return leaf(i, c);
        const int h = w / 2;
        LU2MI_TRY(panel(i, c, h));
        const long off = (long)(c - i);
        if (h <= lu2mi_gemm::BT64) {   // one workgroup per step (see node_steps64_kernel)
            LU2MI_TRY(node_steps(i, c, h));
            LU2MI_TRY(gemm_call<T>(ctx, n - c - h, h, h, -1.0, A + (long)(c + h) * lda + c, lda,
                                   A + (long)c * lda + c + h, lda, 1.0, A + (long)(c + h) * lda + c + h, lda, 0));
            LU2MI_TRY(panel(i, c + h, h));
            steps.inv_c[steps.ninv] = c;
            steps.inv_h[steps.ninv++] = h;
            return LU2MI_OK;
        }
        LU2MI_TRY(node_steps(i, 0, 0));
        // right half of this node: rows [c, c+h) scaled by 1/d, then
        // X = inv(D^-1 L11) * scaled rows, then the rows below
        {
            const long e = (long)h * h;
            hipLaunchKernelGGL(scale_copy_kernel<T>, dim3((unsigned)((e + 255) / 256)), dim3(256), 0, ctx->stream,
                               A, lda, c, c + h, h, h, Prec<T>::invd(ctx), pwbuf);
            LU2MI_CHECK(hipGetLastError());
            LU2MI_TRY(gemm_call<T>(ctx, h, h, h, 1.0, linv + off * nb + off, nb, pwbuf, h, 0.0,
                                   A + (long)c * lda + c + h, lda, 1));
            LU2MI_TRY(gemm_call<T>(ctx, n - c - h, h, h, -1.0, A + (long)(c + h) * lda + c, lda,
                                   A + (long)c * lda + c + h, lda, 1.0, A + (long)(c + h) * lda + c + h, lda, 0));
        }
        LU2MI_TRY(panel(i, c + h, h));
        LU2MI_TRY(node_steps(i, 0, 0));
        // off-diagonal block of the inverse: X21 = -inv22 * L21 * inv11
        {
            LU2MI_TRY(gemm_call<T>(ctx, h, h, h, 1.0, A + (long)(c + h) * lda + c, lda, linv + off * nb + off, nb,
                                   0.0, tmp, h, 0));
            LU2MI_TRY(gemm_call<T>(ctx, h, h, h, -1.0, linv + (off + h) * nb + off + h, nb, tmp, h, 0.0,
                                   linv + (off + h) * nb + off, nb, 1));
        }
        return LU2MI_OK;
    }

    // scratch pointers of block i (per-block copies when the factors are kept)
    void set_block(int i)
    {
        if (linv_all) {
            linv = linv_all + (long)(i / nb) * nb * nb;
            pairs = pairs_all + (long)(i / nb) * 4 * nb;
        } else if (linv_base) {
            linv = linv_base + (long)((i / nb) & 1) * nb * nb;
            pairs = pairs_base + (long)((i / nb) & 1) * 4 * nb;
        }
    }

    // HIP events around one subsystem's launches on the current stream
    // (recorded only with timing on; slot -1 = not recorded)
    int tbegin(int cat, int &slot)
    {
        slot = -1;
        KernelTimer &kt = ctx->tcat[cat];
        if (!ctx->timing_on || kt.used >= kt.cap) return LU2MI_OK;
        slot = kt.used++;
        LU2MI_CHECK(hipEventRecord(kt.ev[2 * slot], ctx->stream));
        return LU2MI_OK;
    }
    int tend(int cat, int slot, double flops, double bytes)
    {
        if (slot < 0) return LU2MI_OK;
        KernelTimer &kt = ctx->tcat[cat];
        LU2MI_CHECK(hipEventRecord(kt.ev[2 * slot + 1], ctx->stream));
        kt.flops[slot] = flops;
        kt.bytes[slot] = bytes;
        return LU2MI_OK;
    }

    int start_panel(int i)
    {
        set_block(i);
        int ts;
        LU2MI_TRY(tbegin(LU2MI_T_PANEL, ts));
        LU2MI_TRY(panel(i, i, nb));
        LU2MI_TRY(node_steps(i, 0, 0));
        return tend(LU2MI_T_PANEL, ts, (double)(n - i) * nb * nb, 0.0);
    }

    // block-level row permutation of columns [c0, c1) with its timing
    int block_perm(int i, int c0, int c1, T *wb, long ldw, bool first = false)
    {
        int ts;
        LU2MI_TRY(tbegin(LU2MI_T_SWAP, ts));
        LU2MI_TRY(rowperm(pairs, pairs + 2 * nb, 2 * nb, c0, c1, 0, 0, n + 1, i, i + nb, wb, ldw, i, i + nb, first));
        return tend(LU2MI_T_SWAP, ts, 0.0, 32.0 * nb * (double)(c1 - c0));
    }

    // U12 of columns [c0, c0+N) = inv(D^-1 L11) * staged rows (lu2.c:511-512)
    int u12(int i, int c0, int N, const T *wb, long ldw)
    {
        int ts;
        LU2MI_TRY(tbegin(LU2MI_T_U12, ts));
        LU2MI_TRY(gemm_call<T>(ctx, nb, N, nb, 1.0, linv, nb, wb, ldw, 0.0, A + (long)i * lda + c0, lda, 1,
                               (sizeof(T) == 8 && ctx->trail_kernel) ? 1 : 0));
        return tend(LU2MI_T_U12, ts, (double)nb * nb * N, 0.0);
    }

    // A22[:, c0 .. c0+N) -= L21 * U12[:, c0 .. c0+N) for block i (lu2.c:580), timed
    int trailing(int i, int c0, int N)
    {
        const int M = n - i - nb;
        int ts;
        LU2MI_TRY(tbegin(LU2MI_T_TRAIL, ts));
        if (sizeof(T) == 4 && ctx->lowp)   // operands rounded to FP16/BF16, FP32 accumulation
            LU2MI_TRY(lu2mi_update16(ctx, ctx->lowp, M, N, nb, (const float *)(A + (long)(i + nb) * lda + i), lda,
                                     (const float *)(A + (long)i * lda + c0), lda,
                                     (float *)(A + (long)(i + nb) * lda + c0), lda));
        else
            LU2MI_TRY(gemm_call<T>(ctx, M, N, nb, -1.0, A + (long)(i + nb) * lda + i, lda, A + (long)i * lda + c0,
                                   lda, 1.0, A + (long)(i + nb) * lda + c0, lda, 0, ctx->trail_kernel ? 1 : 2));
        return tend(LU2MI_T_TRAIL, ts, 2.0 * M * (double)N * nb, 0.0);
    }

    // Block loop of lu2.c:1122-1144.  With lookahead, block i's row
    // permutation, U12 product and trailing update are each split: the next
    // panel's nb columns first, then the rest; the next panel is factored on
    // the second stream as soon as its columns are up to date, while the rest
    // of block i runs.  The two touch disjoint columns; the next panel has its
    // own Linv and pair buffers (they alternate by block) and its own staging
    // rows, so block i's stay intact until its rest is done.
    int run(int *dpiv_out, T *dx)
    {
        const bool la = ctx->lookahead != 0;
        hipStream_t s1 = ctx->stream;
        bool panel_pending = false;   // panel(i) issued on the second stream
        // the inverses' blocks above the diagonal, which nothing writes, zeroed
        // once for all blocks (a launch per block stood before every panel)
        {
            T *const z = linv_all ? linv_all : linv_base;
            const long count = (long)nb * (linv_all ? n : 2 * nb);
            hipLaunchKernelGGL(fill_kernel<T>, dim3(1024), dim3(256), 0, s1, z, count, T(0));
            LU2MI_CHECK(hipGetLastError());
        }
        LU2MI_TRY(start_panel(0));
        for (int i = 0; i < n; i += nb) {
            if (panel_pending) {
                LU2MI_CHECK(hipStreamWaitEvent(s1, ctx->ev_panel, 0));
                panel_pending = false;
            }
            set_block(i);
            const int ncols = n + 1 - (i + nb);
            const int M = n - i - nb;
            const int na = (la && M > 0) ? nb : ncols;   // columns before the split
            // block-level row permutation over [i+nb, n], 1/d scaling of the
            // block rows, block rows staged in w (lu2.c:502-509 awork copy)
            const long ldw = (ncols + 3) & ~3L;   // 16-byte rows for FP64 and FP32
            LU2MI_TRY(block_perm(i, i + nb, i + nb + na, wbuf, ldw, true));
            // U12 = inv(D^-1 L11) * staged rows   (lu2.c:511-512)
            LU2MI_TRY(u12(i, i + nb, na, wbuf, ldw));
            if (M <= 0) continue;
            if (la) {
                LU2MI_TRY(trailing(i, i + nb, nb));                    // the next panel's columns
                LU2MI_CHECK(hipEventRecord(ctx->ev_next, s1));
                // the rest of block i, b included: staging rows from column nb
                // of w on, so that w keeps the layout of the unsplit product.
                // Queued before the panel: a panel is some two hundred
                // launches (n = 32768, nb = 512), and from the middle of the
                // factorization on the device had run them all when the last
                // was queued, with this stream idle beside it: 521 -> 512 ms,
                // n = 49152, nb = 1024 1405 -> 1384 ms, with the panel's
                // kernels at a higher wave priority.
                LU2MI_TRY(block_perm(i, i + 2 * nb, n + 1, wbuf + nb, ldw));
                LU2MI_TRY(u12(i, i + 2 * nb, ncols - nb, wbuf + nb, ldw));
                LU2MI_TRY(trailing(i, i + 2 * nb, ncols - nb));
                LU2MI_CHECK(hipStreamWaitEvent(ctx->stream2, ctx->ev_next, 0));
                ctx->stream = ctx->stream2;                           // panel(i+nb) on the second stream
                const int prc = start_panel(i + nb);
                ctx->stream = s1;
                LU2MI_TRY(prc);
                LU2MI_CHECK(hipEventRecord(ctx->ev_panel, ctx->stream2));
                panel_pending = true;
            } else {
                LU2MI_TRY(trailing(i, i + nb, ncols));
                LU2MI_TRY(start_panel(i + nb));
            }
        }
        if (panel_pending) LU2MI_CHECK(hipStreamWaitEvent(s1, ctx->ev_panel, 0));
        // x = column n, then unit-upper back substitution
        int ts;
        LU2MI_TRY(tbegin(LU2MI_T_BACKSUB, ts));
        hipLaunchKernelGGL(copy_col_kernel<T>, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, A, lda, n, n, dx);
        LU2MI_CHECK(hipGetLastError());
        LU2MI_TRY(backsub(ctx, A, lda, n, dx));
        LU2MI_TRY(tend(LU2MI_T_BACKSUB, ts, (double)n * n, 4.0 * (double)n * n));
        if (dpiv_out && dpiv_out != ctx->d_piv)
            LU2MI_CHECK(hipMemcpyAsync(dpiv_out, ctx->d_piv, sizeof(int) * n, hipMemcpyDeviceToDevice, ctx->stream));
        return LU2MI_OK;
    }
};

template <typename T>
static int factor_impl(lu2mi_ctx *ctx, int n, T *dA, long lda, int nb, int pivmode, int *dpiv_out, T *dx,
                       T *keep_linv = nullptr, int *keep_pairs = nullptr)
{
    if (!ctx || !dA || n <= 0 || lda < n + 1 || nb < 32 || nb > 4096 || (nb & (nb - 1)) || n % nb) {
        lu2mi_set_error_msg("lumcolumn: need nb a power of two in [32, 4096], n %% nb == 0, lda >= n+1 "
                            "(n=%d nb=%d lda=%ld)", n, nb, lda);
        return LU2MI_ERR_ARG;
    }
    LU2MI_TRY(lu2mi_ctx_reserve(ctx, n, nb, sizeof(T)));
    T *x = dx ? dx : (T *)ctx->d_y;
    Factor<T> f;
    f.ctx = ctx; f.A = dA; f.lda = lda; f.n = n; f.nb = nb;
    f.compat = (pivmode == LU2MI_PIV_COMPAT);
    f.W = (ctx->leaf_w == 16) ? 16 : 32;
    if (f.W > nb / 2) f.W = 16;
    // a W=32 leaf holds at most 2 rows per thread in registers over LEAF_GMAX workgroups
    if (f.W == 32 && n > 2 * NTL * LEAF_GMAX) f.W = 16;
    f.linv = (T *)ctx->d_linv; f.tmp = (T *)ctx->d_tmp; f.wbuf = (T *)ctx->d_w; f.pairs = ctx->d_pairs;
    f.pwbuf = (T *)((double *)ctx->d_tmp + (size_t)ctx->nb_cap * ctx->nb_cap);
    f.linv_base = (T *)ctx->d_linv; f.pairs_base = ctx->d_pairs;
    f.linv_all = keep_linv;
    f.pairs_all = keep_pairs;
    for (int c = 0; c < LU2MI_T_COUNT; c++) ctx->tcat[c].used = 0;
    LU2MI_CHECK(hipMemsetAsync(ctx->d_err, 0, sizeof(int), ctx->stream));
    // slot sequence numbers restart with every factorization
    LU2MI_CHECK(hipMemsetAsync(ctx->d_slots, 0, ctx->slots_bytes, ctx->stream));
    ctx->bar_count = 0;
    ctx->gbar_count = 0;
    auto t0 = std::chrono::steady_clock::now();
    int rc = f.run(dpiv_out, x);
    if (rc != LU2MI_OK) return rc;
    LU2MI_CHECK(hipStreamSynchronize(ctx->stream));
    auto t1 = std::chrono::steady_clock::now();
    ctx->t_last_ms[3] = std::chrono::duration<double, std::milli>(t1 - t0).count();
    int herr = 0;
    LU2MI_CHECK(hipMemcpy(&herr, ctx->d_err, sizeof(int), hipMemcpyDeviceToHost));
    if (herr) {
        lu2mi_set_error_msg("leaf kernel grid barrier timed out");
        return LU2MI_ERR_DEVICE;
    }
    return LU2MI_OK;
}

int lu2mi_factor_f64(lu2mi_ctx *ctx, int n, double *dA, long lda, int nb, int pivmode, int *dpiv, double *dx)
{
    return factor_impl<double>(ctx, n, dA, lda, nb, pivmode, dpiv, dx);
}
int lu2mi_factor_f32(lu2mi_ctx *ctx, int n, float *dA, long lda, int nb, int pivmode, int *dpiv, float *dx,
                     float *keep_linv, int *keep_pairs)
{
    return factor_impl<float>(ctx, n, dA, lda, nb, pivmode, dpiv, dx, keep_linv, keep_pairs);
}
int lu2mi_factor_f64_keep(lu2mi_ctx *ctx, int n, double *dA, long lda, int nb, int pivmode, int *dpiv,
                          double *dx, double *keep_linv, int *keep_pairs)
{
    return factor_impl<double>(ctx, n, dA, lda, nb, pivmode, dpiv, dx, keep_linv, keep_pairs);
}
// lu2tlib.c:1130 cm_column_decomposition_recursive on a device copy: the
// panel's rows [i, n) of m columns (column-major, leading dimension ld)
// factored in place with the recursive panel; pv[k] = global pivot row.
int lu2mi_cm_panel_f64(lu2mi_ctx *ctx, double *dcm, long ld, int n, int m, int i, int pivmode, int *hpv)
{
    if (m != 16 && m != 32) {
        lu2mi_set_error_msg("cm panel: %d columns (16 or 32 supported)", m);
        return LU2MI_ERR_UNSUPPORTED;
    }
    const int R = n - i;
    if (R < m) {
        lu2mi_set_error_msg("cm panel: %d rows for %d columns", R, m);
        return LU2MI_ERR_ARG;
    }
    const long ldp = 2 * m;
    LU2MI_TRY(lu2mi_ctx_reserve(ctx, R, 2 * m > 64 ? 2 * m : 64, sizeof(double)));
    double *P = nullptr;
    LU2MI_CHECK(hipMalloc(&P, sizeof(double) * (size_t)R * ldp));
    const long tot = (long)R * m;
    hipLaunchKernelGGL(cm_to_rm_kernel, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, ctx->stream, dcm, ld, i,
                       R, m, P, ldp, 0);
    Factor<double> f;
    f.ctx = ctx; f.A = P; f.lda = ldp; f.n = R; f.nb = m; f.compat = (pivmode == LU2MI_PIV_COMPAT); f.W = m;
    f.linv = (double *)ctx->d_linv; f.tmp = (double *)ctx->d_tmp; f.wbuf = (double *)ctx->d_w;
    f.pwbuf = (double *)ctx->d_tmp + (size_t)ctx->nb_cap * ctx->nb_cap;
    f.pairs = ctx->d_pairs;
    int rc = LU2MI_OK;
    if (hipMemsetAsync(ctx->d_err, 0, sizeof(int), ctx->stream) != hipSuccess ||
        hipMemsetAsync(ctx->d_slots, 0, ctx->slots_bytes, ctx->stream) != hipSuccess)
        rc = LU2MI_ERR_HIP;
    ctx->bar_count = 0;
    ctx->gbar_count = 0;
    if (rc == LU2MI_OK) rc = f.panel(0, 0, m);
    if (rc == LU2MI_OK) rc = f.node_steps(0, 0, 0);
    if (rc == LU2MI_OK) {
        hipLaunchKernelGGL(cm_to_rm_kernel, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, ctx->stream, dcm, ld,
                           i, R, m, P, ldp, 1);
        int piv[32], herr = 0;
        if (hipMemcpyAsync(piv, ctx->d_piv, sizeof(int) * m, hipMemcpyDeviceToHost, ctx->stream) != hipSuccess ||
            hipMemcpyAsync(&herr, ctx->d_err, sizeof(int), hipMemcpyDeviceToHost, ctx->stream) != hipSuccess ||
            hipStreamSynchronize(ctx->stream) != hipSuccess)
            rc = LU2MI_ERR_HIP;
        else if (herr)
            rc = LU2MI_ERR_DEVICE;
        else
            for (int k = 0; k < m; k++) hpv[k] = i + piv[k];
    }
    (void)hipStreamSynchronize(ctx->stream);
    (void)hipFree(P);
    if (rc == LU2MI_ERR_HIP) lu2mi_set_error_msg("cm panel: HIP call failed");
    if (rc == LU2MI_ERR_DEVICE) lu2mi_set_error_msg("cm panel: device wait timed out");
    return rc;
}

int lu2mi_backsub_f32_f64(lu2mi_ctx *ctx, const float *A, long lda, int n, double *x)
{
    return backsub<float, double>(ctx, A, lda, n, x);
}
int lu2mi_backsub_f64_f64(lu2mi_ctx *ctx, const double *A, long lda, int n, double *x)
{
    return backsub<double, double>(ctx, A, lda, n, x);
}

// ---------------------------------------------------------------------------
int lu2mi_randomsetmat_impl(lu2mi_ctx *ctx, int n, int seed, double *dA, long lda)
{
    if (!ctx || !dA || n <= 0 || lda < n + 1) {
        lu2mi_set_error_msg("randomsetmat: bad arguments");
        return LU2MI_ERR_ARG;
    }
    const unsigned long long x0 = (((unsigned long long)(unsigned)seed) << 16) | 0x330EULL;
    hipLaunchKernelGGL(randomsetmat_kernel, dim3(n), dim3(256), 0, ctx->stream, dA, lda, n, x0);
    LU2MI_CHECK(hipGetLastError());
    LU2MI_CHECK(hipStreamSynchronize(ctx->stream));
    return LU2MI_OK;
}

int lu2mi_diag_dominant_impl(lu2mi_ctx *ctx, int n, double *dA, long lda)
{
    if (!dA || n <= 0 || lda < n + 1) {
        lu2mi_set_error_msg("make_diag_dominant: bad arguments");
        return LU2MI_ERR_ARG;
    }
    hipLaunchKernelGGL(diag_dominant_kernel, dim3(n), dim3(256), 0, ctx->stream, dA, lda, n);
    LU2MI_CHECK(hipGetLastError());
    LU2MI_CHECK(hipStreamSynchronize(ctx->stream));
    return LU2MI_OK;
}

// the three residual kernels on ctx's stream: buf holds 3n doubles of
// partial results, dout (device) receives the ten figures
static int residual_launch(lu2mi_ctx *ctx, int n, const double *dA0, long lda, const double *dx, double *buf,
                           double *dout)
{
    double *rerr = buf, *rabs = buf + n, *cabs = buf + 2 * (size_t)n;
    hipLaunchKernelGGL(resid_rows_kernel, dim3((n + 4 * RESID_ROWS - 1) / (4 * RESID_ROWS)), dim3(256), 0, ctx->stream,
                       dA0, lda, n, dx, rerr, rabs);
    hipLaunchKernelGGL(resid_cols_kernel, dim3((n + 63) / 64), dim3(64 * RESID_CW), 0, ctx->stream, dA0, lda, n, cabs);
    hipLaunchKernelGGL(resid_final_kernel, dim3(1), dim3(256), 0, ctx->stream, dA0, lda, n, dx, rerr, rabs, cabs,
                       dout);
    LU2MI_CHECK(hipGetLastError());
    return LU2MI_OK;
}

int lu2mi_residual_impl(lu2mi_ctx *ctx, int n, const double *dA0, long lda, const double *dx, double *out)
{
    if (!ctx || !dA0 || !dx || !out || n <= 0 || lda < n + 1) {
        lu2mi_set_error_msg("residual: bad arguments");
        return LU2MI_ERR_ARG;
    }
    double *buf = nullptr;
    LU2MI_CHECK(hipMalloc(&buf, sizeof(double) * (3 * (size_t)n + 16)));
    int rc = residual_launch(ctx, n, dA0, lda, dx, buf, buf + 3 * (size_t)n);
    hipError_t e = hipSuccess;
    if (rc == LU2MI_OK) {
        e = hipMemcpyAsync(out, buf + 3 * (size_t)n, 10 * sizeof(double), hipMemcpyDeviceToHost, ctx->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    }
    (void)hipFree(buf);
    if (rc != LU2MI_OK) return rc;
    if (e != hipSuccess) {
        lu2mi_set_error_msg("residual: %s", hipGetErrorString(e));
        return LU2MI_ERR_HIP;
    }
    return LU2MI_OK;
}

// address of this device's copy of scratch (called once per device, with the
// device current, when a context is created)
int lu2mi_scratch_address(double **p)
{
    *p = nullptr;
    LU2MI_CHECK(hipGetSymbolAddress((void **)p, HIP_SYMBOL(scratch)));
    return LU2MI_OK;
}

int lu2mi_residual_noalloc_impl(lu2mi_ctx *ctx, int n, const double *dA0, long lda, const double *dx, double *dout)
{
    if (!ctx || !dA0 || !dx || !dout || n <= 0 || lda < n + 1) {
        lu2mi_set_error_msg("residual (no allocation): bad arguments");
        return LU2MI_ERR_ARG;
    }
    if (n > LU2MI_RESID_NMAX) {
        lu2mi_set_error_msg("residual (no allocation): n = %d exceeds the scratch limit %d", n, LU2MI_RESID_NMAX);
        return LU2MI_ERR_ARG;
    }
    if (!ctx->d_scratch) {
        lu2mi_set_error_msg("residual (no allocation): scratch address unknown");
        return LU2MI_ERR_HIP;
    }
    return residual_launch(ctx, n, dA0, lda, dx, ctx->d_scratch, dout);
}
