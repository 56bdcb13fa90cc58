// Device code of libpizza_amd: the dense inversions of the collocation
// method's matrix rebuilds.  Included by pz_coll.h.
#pragma once
#include "pz_device.h"

typedef double pz_d4 __attribute__((ext_vector_type(4)));

#define GJ_B 16      // pivot columns per panel: the k extent of the update's tiles
#define GJ_NMAX 512  // largest order (the row index takes 9 bits of the pivot key)
#define GJ_ROWW 8    // waves that hold the rows of a panel at GJ_NMAX
// pivot columns a row keeps in registers at a time (32 registers): a panel
// of complex columns is two of these, merged behind the second
template <class M> constexpr int gj_sub() { return sizeof(M) == 8 ? 16 : 8; }

// LDS of gj_invert (16-byte blocks): U [GJ_B][np] with np = n rounded up to
// 16, the pivot rows of a column chunk Wk [GJ_B][cw], the waves' pivot
// candidates of two steps (row and reciprocal) and their keys, the pivot row
// of each step, the slots of the finished columns that are wanted, the slots
// of a chunk's columns and a flag for the panel's pivot rows.
template <class M>
struct GjLayout {
    size_t U, Wk, cand, key, perm, done, col, piv, total;
    int np, cw;
    __host__ __device__ GjLayout(int n)
    {
        size_t o = 0;
        auto take = [&](size_t bytes) { size_t r = o; o += (bytes + 15) & ~(size_t)15; return r; };
        np = (n + 15) & ~15;
        // the widest chunk whose pivot rows fit next to U at n = 512 (complex)
        cw = n <= 384 ? 128 : 32;
        U = take(sizeof(M) * GJ_B * np);
        Wk = take(sizeof(M) * GJ_B * cw);
        cand = take(sizeof(M) * 2 * GJ_ROWW * (gj_sub<M>() + 1));
        key = take(sizeof(double) * 2 * GJ_ROWW);
        perm = take(sizeof(short) * np);
        done = take(sizeof(short) * np);
        col = take(sizeof(short) * cw);
        piv = take(sizeof(short) * np);
        total = o;
    }
};
template <class M>
__host__ __device__ inline size_t gj_lds_bytes(int n) { return GjLayout<M>(n).total; }

// the largest of a wave's non-negative values (uniform): row shifts within
// 16 lanes, then the two row broadcasts, all on the vector unit
template <int CTRL, int ROWS> __device__ __forceinline__ double gj_dpp_max(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xF, false);
    return fmax(v, __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo));
}
__device__ __forceinline__ double gj_wave_max(double v)
{
    v = gj_dpp_max<0x111, 0xF>(v); // row_shr:1, 2, 4, 8
    v = gj_dpp_max<0x112, 0xF>(v);
    v = gj_dpp_max<0x114, 0xF>(v);
    v = gj_dpp_max<0x118, 0xF>(v);
    v = gj_dpp_max<0x142, 0xA>(v); // row_bcast:15 into rows 1 and 3
    v = gj_dpp_max<0x143, 0xC>(v); // row_bcast:31 into rows 2 and 3
    return rl(v, 63);
}

// 1 / a, the larger part divided first (Smith) without a branch
__device__ __forceinline__ double gj_recip(double a) { return 1.0 / a; }
__device__ __forceinline__ cd gj_recip(cd a)
{
    const bool sw = fabs(a.x) < fabs(a.y);
    const double g = sw ? a.y : a.x, h = sw ? a.x : a.y, r = h / g, d = 1.0 / (g + h * r), e = -r * d;
    return sw ? mk(-e, -d) : mk(d, e);
}

// acc += A B on one 16 x 16 tile of 4 k values (v_mfma_f64_16x16x4): lane l
// gives A[l % 16][l / 16] and B[l / 16][l % 16] and holds rows l / 16 + 4 r,
// column l % 16 of acc
__device__ __forceinline__ pz_d4 gj_mfma(double a, double b, pz_d4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// the 16 x 16 tile of one wave: acc += U[i0 .., 0..15] Wk[0..15, j ..]
__device__ __forceinline__ void gj_tile(const double *U, int np, const double *Wk, int cw, int i0, int jt, double (&w)[4])
{
    const int lane = threadIdx.x & 63, i = lane & 15, k = lane >> 4;
    pz_d4 acc = {w[0], w[1], w[2], w[3]};
#pragma unroll
    for (int s = 0; s < GJ_B / 4; s++) acc = gj_mfma(U[(4 * s + k) * np + i0 + i], Wk[(4 * s + k) * cw + jt + i], acc);
#pragma unroll
    for (int r = 0; r < 4; r++) w[r] = acc[r];
}
__device__ __forceinline__ void gj_tile(const cd *U, int np, const cd *Wk, int cw, int i0, int jt, cd (&w)[4])
{
    const int lane = threadIdx.x & 63, i = lane & 15, k = lane >> 4;
    pz_d4 re = {w[0].x, w[1].x, w[2].x, w[3].x}, im = {w[0].y, w[1].y, w[2].y, w[3].y};
#pragma unroll
    for (int s = 0; s < GJ_B / 4; s++) {
        const cd u = U[(4 * s + k) * np + i0 + i], v = Wk[(4 * s + k) * cw + jt + i];
        re = gj_mfma(u.x, v.x, re);
        im = gj_mfma(u.x, v.y, im);
        re = gj_mfma(-u.y, v.y, re);
        im = gj_mfma(u.y, v.x, im);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) w[r] = mk(re[r], im[r]);
}

// The first panel of the omega-psi system.  Its omega block has N columns and
// only N - 2 omega equations (two of its rows are wall conditions on psi), so
// the pivots N - 2 and N - 1 (counted from 0) come from the rows of omega =
// -Laplacian(psi), whose omega entries the row scaling leaves at 1e-6.  A group
// of pivot columns that ends between the two has coefficients U of 1e6, and the
// columns behind it, formed as U W[K], lose that factor where the
// column-by-column elimination does not: at n_r 9 the residual of a solve was
// up to 128 times that of an elimination without panels, at n_r 17 7 times.
// Groups of 8 end there when N - 1 is a multiple of 8; four columns first put
// both pivots inside a group (2.1 and 2.7 times).  From n_r 25 on the loss is
// lost in the spread between orders of elimination (up to 5 times with either
// panel, and 20 times at n_r 145 with four columns first in one of eight runs),
// so the whole panel stays.  2 N is 2 more than a multiple of 16 there: the
// number of panels is the same.
__host__ __device__ constexpr int gj_first_psi(int N) { return N <= 17 && (N - 1) % 8 == 0 ? 4 : GJ_B; }

// In-place blocked Gauss-Jordan inversion with partial pivoting of the
// row-major n x n block W by one workgroup of 1024 threads, forming only the
// columns of A^{-1} that multiply the first nr entries of a right-hand side.
// No rows are swapped: perm[k] is the row of pivot k, and on return
//     A^{-1}[k][perm[s]] = W[perm[k]][s]   for perm[s] < nr.
// The pivot columns live in registers, one row per thread: step q takes the
// largest |re| + |im| of column q among the rows without a pivot (the row
// index in the low bits of the compared value settles ties, first row
// first), each wave offers its best row, and one barrier later every thread
// adds -f_i / p times the pivot row to its row (1 / p times it for the pivot
// row itself), in the columns still to come and, as the columns behind it
// turn into the coefficients U of the panel's pivot rows, in those.  A row i
// outside the panel's pivot rows K is then W_i + U_i W[K], a pivot row
// U_i W[K] (not W_i + (1 / p - 1) W_i, which would lose the digits of 1 / p at
// large pivots).  Two groups of complex columns compose to U_1 + U_2 U_1[K_2]
// (without U_1 in the rows K_2) and U_2.  The other columns get this update
// in one pass of 16 x 16 tiles on the matrix cores, and the panel's slots take
// U, the inverse's columns so far.
// What bounds it: the pivot steps' serial chain (one barrier each) at small
// n; the passes over W, n^2 / 16 times the matrix, at large n.  In place the
// blocks of all modes stay in the last-level cache (181 MB at n = 258 and 170
// modes, where [A | I] took 362 MB), and finished columns that the m-loop
// does not apply drop out of the passes (a quarter of the work for psi).
// Measured, k_build_coll at n_r 129 and 171 modes: 2.1 ms (5.0 ms with the
// panels and the rank-16 update on the vector unit in LDS, rows swapped); at
// n_r 49 and 49 modes 0.24 ms (0.65 ms).
// first: columns of the first panel, 1 .. GJ_B (gj_first_psi).
// lds: gj_lds_bytes<M>(n).  Returns the LAPACK-style info (k + 1 of the first
// zero pivot, 0 if none).
template <class M>
__device__ int gj_invert(M *W, int n, int nr, char *lds, int first = GJ_B)
{
    constexpr int SB = gj_sub<M>();
    const GjLayout<M> lay(n);
    const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63, wave = tid >> 6, nw = nt >> 6;
    const int np = lay.np, cw = lay.cw, rw = (n + 63) >> 6; // waves that hold rows
    M *U = (M *)(lds + lay.U), *Wk = (M *)(lds + lay.Wk), *cand = (M *)(lds + lay.cand);
    double *key = (double *)(lds + lay.key);
    short *perm = (short *)(lds + lay.perm), *done = (short *)(lds + lay.done), *col = (short *)(lds + lay.col);
    short *piv = (short *)(lds + lay.piv);
    const bool row = tid < n, holds = wave < rw;
    bool used = false; // this thread's row has been a pivot row
    int ndone = 0;     // finished columns that are wanted (slots in done)
    if (tid < 2 * GJ_ROWW) key[tid] = 0.0;
    __syncthreads();
    for (int k0 = 0, b; k0 < n; k0 += b) {
        b = min(k0 == 0 ? first : GJ_B, n - k0);
        bool inpanel = false; // this thread's row is a pivot row of the panel
        for (int s0 = 0; s0 < b; s0 += SB) {
            const int k1 = k0 + s0, bs = min(SB, b - s0);
            M v[SB];
#pragma unroll
            for (int c = 0; c < SB; c++) v[c] = row && c < bs ? W[(size_t)tid * n + k1 + c] : mzero<M>();
            if (s0 > 0) {
                // the earlier groups of this panel: v += U W[K, k1 ..]
                for (int t = tid; t < s0 * SB; t += nt) {
                    const int q = t / SB, c = t - q * SB;
                    Wk[t] = c < bs ? W[(size_t)perm[k0 + q] * n + k1 + c] : mzero<M>();
                }
                __syncthreads();
                if (inpanel)
#pragma unroll
                    for (int c = 0; c < SB; c++) v[c] = mzero<M>();
                if (row)
                    for (int q = 0; q < s0; q++) {
                        const M u = U[q * np + tid];
#pragma unroll
                        for (int c = 0; c < SB; c++) v[c] = madd(v[c], mmm(u, Wk[q * SB + c]));
                    }
            }
            int info = 0;
            bool ingroup = false;
#pragma unroll
            for (int q = 0; q < SB; q++) {
                if (q < bs && info == 0) { // uniform
                    M *cq = cand + (size_t)((q & 1) * GJ_ROWW) * (SB + 1);
                    double *kq = key + (q & 1) * GJ_ROWW;
                    if (holds) {
                        const double a = mabs1(v[q]);
                        const double mine = row && !used && a > 0.0
                                                ? __longlong_as_double((__double_as_longlong(a) & ~(long long)(GJ_NMAX - 1)) |
                                                                       (long long)(GJ_NMAX - 1 - tid))
                                                : 0.0;
                        const M rp = gj_recip(v[q]);
                        const double best = gj_wave_max(mine);
                        M *o = cq + wave * (SB + 1);
                        if (mine == best && best > 0.0) {
#pragma unroll
                            for (int s = 0; s < SB; s++) o[s] = v[s];
                            o[SB] = rp;
                        }
                        if (lane == 0) kq[wave] = best;
                    }
                    __syncthreads();
                    double best = kq[0];
#pragma unroll
                    for (int w = 1; w < GJ_ROWW; w++) best = fmax(best, kq[w]);
                    if (best == 0.0) {
                        info = k1 + q + 1;
                    } else {
                        const int pr = GJ_NMAX - 1 - (int)(__double_as_longlong(best) & (GJ_NMAX - 1));
                        if (tid == 0) perm[k1 + q] = (short)pr;
                        if (holds) {
                            const M *o = cq + (pr >> 6) * (SB + 1);
                            const M rp = o[SB];
                            const bool is = tid == pr;
                            ingroup |= is;
                            used |= is;
                            const M c = is ? rp : mneg(mmm(v[q], rp));
#pragma unroll
                            for (int s = 0; s < SB; s++)
                                if (s != q) v[s] = madd(is ? mzero<M>() : v[s], mmm(c, o[s]));
                            v[q] = c;
                        }
                    }
                }
            }
            __syncthreads();
            if (info) return info;
            if (s0 > 0) {
                // U_1 += U_2 U_1[K_2]
                for (int t = tid; t < s0 * bs; t += nt) {
                    const int s = t / bs, q = t - s * bs;
                    Wk[s * SB + q] = U[s * np + perm[k1 + q]];
                }
                __syncthreads();
                if (row)
                    for (int s = 0; s < s0; s++) {
                        M u = ingroup ? mzero<M>() : U[s * np + tid];
#pragma unroll
                        for (int q = 0; q < SB; q++)
                            if (q < bs) u = madd(u, mmm(v[q], Wk[s * SB + q]));
                        U[s * np + tid] = u;
                    }
            }
            inpanel |= ingroup;
            if (tid < np) {
#pragma unroll
                for (int q = 0; q < SB; q++) U[(s0 + q) * np + tid] = q < bs && row ? v[q] : mzero<M>();
            }
        }
        // columns of U beyond a short last panel
        if (tid < np)
            for (int s = (b + SB - 1) / SB * SB; s < GJ_B; s++) U[s * np + tid] = mzero<M>();
        if (tid < np) piv[tid] = inpanel;
        // the inverse's columns so far to the panel's slots
        if (row)
            for (int s = 0; s < b; s++)
                if (perm[k0 + s] < nr) W[(size_t)tid * n + k0 + s] = U[s * np + tid];
        // W[:, J] += U W[K, J] (pivot rows: U W[K, J]) over the finished columns that are wanted and
        // the columns to come, cw at a time
        const int nl = n - k0 - b, nJ = ndone + nl, nrt = np >> 4;
        for (int j0 = 0; j0 < nJ; j0 += cw) {
            const int wc = min(cw, nJ - j0), ct = (wc + 15) >> 4;
            for (int t = tid; t < wc; t += nt) {
                const int jj = j0 + t;
                col[t] = (short)(jj < ndone ? done[jj] : k0 + b + (jj - ndone));
            }
            __syncthreads();
            for (int t = tid; t < GJ_B * 16 * ct; t += nt) {
                const int q = t / (16 * ct), jc = t - q * 16 * ct;
                Wk[q * cw + jc] = q < b && jc < wc ? W[(size_t)perm[k0 + q] * n + col[jc]] : mzero<M>();
            }
            __syncthreads();
            const int jl = lane & 15, il = lane >> 4;
            for (int t = wave; t < nrt * ct; t += nw) {
                const int it = t / ct, jt = t - it * ct, jc = 16 * jt + jl;
                const bool in = jc < wc;
                M *wp = W + (in ? (int)col[jc] : 0);
                M w[4];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int i = 16 * it + il + 4 * r;
                    w[r] = in && i < n && !piv[i] ? wp[(size_t)i * n] : mzero<M>();
                }
                gj_tile(U, np, Wk, cw, 16 * it, 16 * jt, w);
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int i = 16 * it + il + 4 * r;
                    if (in && i < n) wp[(size_t)i * n] = w[r];
                }
            }
            __syncthreads();
        }
        __syncthreads();
        // the panel's wanted slots join the finished ones (every thread
        // counts them; the entries are written by one)
        for (int s = 0; s < b; s++)
            if (perm[k0 + s] < nr) {
                if (tid == 0) done[ndone] = (short)(k0 + s);
                ndone++;
            }
        __syncthreads();
    }
    return 0;
}
