// Device code of libpizza_amd, part 2: the per-m stage kernel (explicit
// assembly + implicit solves of the integration method), the start-up
// kernel, diagnostics and unit-operator kernels.  Included once by pz_api.hip.
#pragma once
#include "pz_device.h"

// set_imex_rhs for one m row (multistep_schemes.f90:366-413;
// dirk_schemes.f90:773-814), split around the current explicit slot: P sums
// (in the reference's order) every term before it, Q every term after it, and the
// right-hand side is (P + w cur) + Q with w = imex_weight().  Lets the
// global-memory terms be loaded and summed before cur is known.
__device__ __forceinline__ void imex_split(const PzDev &p, const PzScheme *s, int istage, const cd *old,
                                           const cd *impl, const cd *expl, size_t off, int k, cd &P, cd &Q)
{
    const size_t F = (size_t)p.nm * p.N;
    const int is = istage - 1;
    cd r, q = mk(0.0, 0.0);
    if (p.family == 0) {
        r = cscale(s->wimp[0], gld(old, off + k));
        for (int o = 1; o < p.nold; o++) r = cadd(r, cscale(s->wimp[o], gld(old, o * F + off + k)));
        for (int o = 0; o < p.nimp; o++) r = cadd(r, cscale(s->wimp_lin[o + 1], gld(impl, o * F + off + k)));
        for (int o = 0; o < is; o++) r = cadd(r, cscale(s->wexp[o], gld(expl, o * F + off + k)));
        for (int o = is + 1; o < p.nexp; o++) {
            const cd t = cscale(s->wexp[o], gld(expl, o * F + off + k));
            q = o == is + 1 ? t : cadd(q, t);
        }
    } else {
        r = gld(old, off + k);
        for (int st = 0; st < is; st++) r = cadd(r, cscale(s->bexp[istage][st], gld(expl, st * F + off + k)));
        for (int st = 0; st <= is; st++) {
            const cd t = cscale(s->bimp[istage][st], gld(impl, st * F + off + k));
            q = st == 0 ? t : cadd(q, t);
        }
    }
    P = r;
    Q = q;
}
__device__ __forceinline__ double imex_weight(const PzDev &p, const PzScheme *s, int istage)
{
    return p.family == 0 ? s->wexp[istage - 1] : s->bexp[istage][istage - 1];
}

// -BuoFac rgrav/r i m T - ChemFac rgrav/r i m X (update_psi_integ_smat.f90:286-304)
__device__ __forceinline__ cd buoyancy(const PzDev &p, const RadView &R, int m, int k, cd T, cd X)
{
    cd b = mk(0, 0);
    if (m == 0) return b;
    if (p.l_heat) {
        double s = -p.BuoFac * R.rgrav(k) * R.or1(k);
        b = cmul(mk(0.0, s * (double)m), T);
        if (p.l_chem) b = csub(b, cmul(mk(0.0, p.ChemFac * R.rgrav(k) * R.or1(k) * (double)m), X));
    } else if (p.l_chem) {
        double s = -p.ChemFac * R.rgrav(k) * R.or1(k);
        b = cmul(mk(0.0, s * (double)m), X);
    }
    return b;
}

// get_dcheb_real_1d with the rerror threshold (radial_derivatives.f90:143-185),
// one thread: Chebyshev coefficients of d/dx from those of f
__device__ __forceinline__ void dcheb_real(const PzDev &p, const double *__restrict__ f, double *__restrict__ df)
{
    const int N = p.N;
    // four independent maxima so that the loads overlap
    double m0 = 0.0, m1 = 0.0, m2 = 0.0, m3 = 0.0;
    int j = 0;
    for (; j + 3 < N; j += 4) {
        m0 = fmax(m0, fabs(f[j]));
        m1 = fmax(m1, fabs(f[j + 1]));
        m2 = fmax(m2, fabs(f[j + 2]));
        m3 = fmax(m3, fabs(f[j + 3]));
    }
    for (; j < N; j++) m0 = fmax(m0, fabs(f[j]));
    const double thr = fmax(fmax(m0, m1), fmax(m2, m3)) * p.thr;
    // the recurrence df(n-1) = df(n+1) + 2 n f(n) carried in registers:
    // up1 = df(n), up2 = df(n+1)
    df[N - 1] = 0.0;
    const int nc = N - 1;
    double up1 = fabs(f[nc]) >= thr ? (double)nc * f[nc] : 0.0, up2 = 0.0;
    df[nc - 1] = up1;
#pragma unroll 4
    for (int n = N - 2; n >= 1; n--) {
        const double fn = f[n];
        const double v = fabs(fn) >= thr ? up2 + (double)(2 * n) * fn : 0.0;
        df[n - 1] = v;
        up2 = up1;
        up1 = v;
    }
}

#define MPHASE_NVEC 24
#define PZ_MPHASE_THREADS 512
// threads of the m-loop kernels for n_r: 256 leave room for more
// workgroups per CU on small grids (the coupled collocation system needs
// 2 n_r <= threads)
__host__ __device__ constexpr int mloop_threads(int N) { return N <= 65 ? 256 : PZ_MPHASE_THREADS; }

// column groups of a product with `threads` threads: the partial sums of three
// vectors must fit the kernel's reduction scratch
__host__ __device__ constexpr int shared_groups(int N, int threads)
{
    const int rq = (N + 3) / 4, cap = N <= 160 ? 8 : 3;
    int cg = threads / rq;
    if (cg > cap) cg = cap;
    return cg < N ? cg : N;
}

// complex values of an m-loop kernel's scratch `red`: the FFT buffers of the
// Chebyshev transforms (6 L + 12), shared with the partial sums of the dense
// products.  Each product a kernel may run is listed with the rows, columns
// and rows a thread it is called with: block_matvec keeps the sums of all
// column groups but the first in registers (matvec_scratch), MatAhead stores
// those of every group (ahead_scratch), SharedMv [vector][group][n_r rounded
// up to 4], with half the threads for T and xi and half for psi.
constexpr size_t mloop_scratch(int N, int threads, bool integ)
{
    const size_t ldm = (N + 3) & ~3;
    const size_t need[] = {6 * (2 * (size_t)N - 2) + 16,
                           matvec_scratch(N, N, threads, 2, 2),     // T and xi
                           matvec_scratch(N, N, threads, 1, 1),
                           matvec_scratch(2 * N, N, threads, 1, 1), // omega and psi
                           // T, xi: one ahead (collocation), both (integration)
                           ahead_scratch(N, N, threads, 2, integ ? 2 : 1),
                           ahead_scratch(integ ? N : 2 * N, N, threads, 1, 1),
                           integ ? 3 * shared_groups(N, threads / 2) * ldm : 0,
                           integ ? shared_groups(N, threads) * ldm : 0};
    size_t most = 0;
    for (size_t n : need) most = n > most ? n : most;
    return most;
}

// LDS layout of the m-loop kernels: working vectors, transform tables and, up
// to the end of the launch's LDS (mloop_lds), the scratch red (16-byte aligned
// blocks).  The kernels compute the offsets, inlined; the size of red is the
// host's (computed in the kernels, its list of products takes scratch memory and
// registers there: fifty BPR353 steps at n_r 97 12.06 ms, 11.73 ms without).
struct MpLayout {
    size_t vec = 0, cosT = 0, sinT = 0, rad = 0, red = 0;
    // rad_lds = false: the radial rows and the transform tables stay in
    // global memory (read through L2), which frees PZ_NRADC n_r + 2 L
    // doubles of LDS per workgroup (collocation m-loop only)
    __host__ __device__ __forceinline__ constexpr MpLayout(int N, bool rad_lds = true)
    {
        size_t o = 0;
        auto take = [&](size_t bytes) { size_t r = o; o += (bytes + 15) & ~(size_t)15; return r; };
        const int L = 2 * N - 2;
        vec = take(sizeof(cd) * MPHASE_NVEC * N);
        // one block [cos L | sin L | radial rows], as in global memory
        cosT = rad_lds ? take(sizeof(double) * (2 * L + PZ_NRADC * N)) : 0;
        sinT = cosT + sizeof(double) * L;
        rad = cosT + sizeof(double) * 2 * L;
        red = o;
    }
};
// bytes of LDS that a launch of an m-loop kernel asks for
constexpr size_t mloop_lds(int N, int threads, bool rad_lds = true, bool integ = false)
{
    return MpLayout(N, rad_lds).red + sizeof(cd) * mloop_scratch(N, threads, integ);
}


// The slots of one field at one point that its right-hand side reads: all of
// them loaded before any is used (imex_split's loops over a run-time number
// of stages wait for each load in turn), summed in imex_split's order, and,
// for a multistep scheme, moved up by one (rotate_imex,
// multistep_schemes.f90:462-498) from the values read: old and impl, the
// explicit slots from the third on; explicit slot 1 takes the current terms
// once they are known (rotate_current).
struct ImexSlots {
    cd o[4], i[4], e[4];
    __device__ __forceinline__ void load(const PzDev &p, int istage, const cd *old, const cd *impl, const cd *expl, size_t q)
    {
        const size_t F = (size_t)p.nm * p.N;
        const int is = istage - 1, ms = p.family == 0;
        // multistep schemes keep at most four slots of each kind
        const int no = ms ? p.nold : 1, ni = ms ? p.nimp : istage, e0 = ms ? 1 : 0, ne = ms ? p.nexp : is;
        const cd z = mk(0.0, 0.0);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            o[k] = k < no ? gld(old, k * F + q) : z;
            i[k] = k < ni ? gld(impl, k * F + q) : z;
            e[k] = k >= e0 && k < ne ? gld(expl, k * F + q) : z;
        }
    }
    __device__ __forceinline__ void sum(const PzDev &p, const PzScheme *s, int istage, cd *old, cd *impl, cd *expl, size_t q,
                                        cd &P, cd &Q) const
    {
        const size_t F = (size_t)p.nm * p.N;
        const int is = istage - 1;
        if (p.family == 0) {
            P = cscale(s->wimp[0], o[0]);
            Q = mk(0.0, 0.0);
#pragma unroll
            for (int k = 1; k < 4; k++)
                if (k < p.nold) P = cadd(P, cscale(s->wimp[k], o[k]));
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (k < p.nimp) P = cadd(P, cscale(s->wimp_lin[k + 1], i[k]));
#pragma unroll
            for (int k = 1; k < 4; k++)
                if (k < p.nexp) Q = k == 1 ? cscale(s->wexp[k], e[k]) : cadd(Q, cscale(s->wexp[k], e[k]));
#pragma unroll
            for (int k = 3; k >= 1; k--) {
                if (k < p.nold) old[k * F + q] = o[k - 1];
                if (k < p.nimp) impl[k * F + q] = i[k - 1];
                if (k >= 2 && k < p.nexp) expl[k * F + q] = e[k - 1];
            }
        } else {
            P = o[0];
            Q = cscale(s->bimp[istage][0], i[0]);
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (k < is) P = cadd(P, cscale(s->bexp[istage][k], e[k]));
#pragma unroll
            for (int k = 1; k < 4; k++)
                if (k <= is) Q = cadd(Q, cscale(s->bimp[istage][k], i[k]));
            for (int k = 4; k < is; k++) P = cadd(P, cscale(s->bexp[istage][k], gld(expl, k * F + q)));
            for (int k = 4; k <= is; k++) Q = cadd(Q, cscale(s->bimp[istage][k], gld(impl, k * F + q)));
        }
    }
};
__device__ __forceinline__ void rotate_current(const PzDev &p, cd *expl, size_t off, int k, cd e)
{
    if (p.family == 0 && p.nexp > 1) expl[(size_t)p.nm * p.N + off + k] = e;
}

// Products with a matrix that all modes share (read through L2, column-major
// [ncol][ldm], ldm = n_r rounded up to 4): rows 4 ru .. 4 ru + 3 and columns
// cg, cg + CG, ... of a thread, for NV vectors at once; four rows a thread,
// since the vectors' LDS reads (one a column) are what the products cost most.
// The first U columns are loaded by load(), and each further batch before the
// one in hand is used.  All groups' partial sums go to red, [vector][CG][ldm].
template <int U> struct SharedMv {
    double2 v[U][2];
    __device__ __forceinline__ void fetch(double2 (&w)[U][2], const double *__restrict__ M, int ldm, int ncol, int cg, int ru,
                                          int CG, int jb) const
    {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int j = cg + (jb + u) * CG;
            const double *q = M + (size_t)j * ldm + 4 * ru;
            w[u][0] = j < ncol ? gld2(q) : mk(0.0, 0.0);
            w[u][1] = j < ncol ? gld2(q + 2) : mk(0.0, 0.0);
        }
    }
    __device__ __forceinline__ void load(const double *__restrict__ M, int ldm, int ncol, int cg, int ru, int CG)
    {
        fetch(v, M, ldm, ncol, cg, ru, CG, 0);
    }
    template <int NV>
    __device__ __forceinline__ void use(const double2 (&w)[U][2], int ncol, const cd *x0, const cd *x1, int cg, int CG, int jb,
                                        cd (&acc)[NV][4]) const
    {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int j = min(cg + (jb + u) * CG, ncol - 1); // columns past the end were loaded as zeros
#pragma unroll
            for (int a = 0; a < NV; a++) {
                const cd x = lds_load(a == 0 ? x0 : x1, j);
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    acc[a][2 * h] = mk(fma(w[u][h].x, x.x, acc[a][2 * h].x), fma(w[u][h].x, x.y, acc[a][2 * h].y));
                    acc[a][2 * h + 1] = mk(fma(w[u][h].y, x.x, acc[a][2 * h + 1].x), fma(w[u][h].y, x.y, acc[a][2 * h + 1].y));
                }
            }
        }
    }
    template <int NV>
    __device__ __forceinline__ void run(const double *__restrict__ M, int ldm, int ncol, const cd *x0, const cd *x1, int cg, int ru,
                                        int CG, cd *red)
    {
        cd acc[NV][4];
#pragma unroll
        for (int a = 0; a < NV; a++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[a][r] = mk(0.0, 0.0);
        const int nj = (ncol - cg + CG - 1) / CG;
        double2 w[U][2];
        for (int jb = 0; jb < nj; jb += 2 * U) {
            if (jb + U < nj) fetch(w, M, ldm, ncol, cg, ru, CG, jb + U);
            use<NV>(v, ncol, x0, x1, cg, CG, jb, acc);
            if (jb + U >= nj) break;
            if (jb + 2 * U < nj) fetch(v, M, ldm, ncol, cg, ru, CG, jb + 2 * U);
            use<NV>(w, ncol, x0, x1, cg, CG, jb + U, acc);
        }
#pragma unroll
        for (int a = 0; a < NV; a++)
#pragma unroll
            for (int r = 0; r < 4; r++) lds_store(red, (a * CG + cg) * ldm + 4 * ru + r, acc[a][r]);
    }
};
// row k of such a product
__device__ __forceinline__ cd shared_sum(const cd *red, int CG, int ldm, int k)
{
    cd s = lds_load(red, k);
    for (int c = 1; c < CG; c++) s = cadd(s, lds_load(red, c * ldm + k));
    return s;
}
// dcheb_real for the real parts of coefficients x in LDS by the first two
// waves of a workgroup (every lane of them calls it): the recurrence
// df(n-1) = df(n+1) + 2 n f(n) links every second coefficient, so each wave
// takes one parity; a lane reduces its elements to an affine map of the value
// entering them (zero where the threshold resets it), a scan over the lanes
// composes the maps, and the lane runs its elements again from what the scan
// hands it.  One lane alone takes 3.6 us at n_r 97.
__device__ __forceinline__ void dcheb_waves(const PzDev &p, const cd *x, cd *df)
{
    const int N = p.N, lane = threadIdx.x & 63, c = threadIdx.x >> 6;
    double thr = 0.0;
    if (p.thr != 0.0) {
        for (int j = lane; j < N; j += 64) thr = fmax(thr, fabs(lds_load(x, j).x));
        for (int o = 32; o > 0; o >>= 1) thr = fmax(thr, __shfl_xor(thr, o, 64));
        thr *= p.thr;
    }
    const int len = (N - c) >> 1, C = (len + 63) >> 6, e0 = lane * C, e1 = min(len, e0 + C);
    double a = 1.0, g = 0.0;
    for (int e = e0; e < e1; e++) {
        const int n = N - 1 - c - 2 * e;
        const double f = lds_load(x, n).x, w = n == N - 1 ? (double)n : (double)(2 * n);
        if (fabs(f) >= thr) {
            g += w * f;
        } else {
            g = 0.0;
            a = 0.0;
        }
    }
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
        const double ap = __shfl_up(a, s, 64), gp = __shfl_up(g, s, 64);
        if (lane >= s) {
            g += a * gp;
            a *= ap;
        }
    }
    double y = __shfl_up(g, 1, 64);
    if (lane == 0) y = 0.0;
    for (int e = e0; e < e1; e++) {
        const int n = N - 1 - c - 2 * e;
        const double f = lds_load(x, n).x, w = n == N - 1 ? (double)n : (double)(2 * n);
        y = fabs(f) >= thr ? y + w * f : 0.0;
        lds_store(df, n - 1, mk(y, 0.0));
    }
    if (c == 0 && lane == 0) lds_store(df, N - 1, mk(0.0, 0.0));
}

// The band coefficients of one row of an m /= 0 mode that the implicit terms
// apply to T, xi and psi, four lanes a row as in bandmv, loaded ahead of the
// transforms of the same phase.
struct BandRow {
    double e2[3], ti[2], pi[5];
    cd pl[5];
    __device__ __forceinline__ void load(const PzDev &p, int mi, int i)
    {
        const int N = p.N, sub = threadIdx.x & 3;
        const bool in = i < N;
        const size_t r = in ? i : 0;
        auto at = [&](int W, int d) { return in && d < W ? d : 0; };
#pragma unroll
        for (int u = 0; u < 3; u++) e2[u] = gld(p.T_RHSE2, r * 9 + at(9, sub + 4 * u));
#pragma unroll
        for (int u = 0; u < 2; u++) ti[u] = gld(p.T_RHSI, ((size_t)mi * N + r) * 5 + at(5, sub + 4 * u));
#pragma unroll
        for (int u = 0; u < 5; u++) pi[u] = gld(p.P_RHSI, ((size_t)mi * N + r) * 17 + at(17, sub + 4 * u));
#pragma unroll
        for (int u = 0; u < 5; u++) pl[u] = gld(p.P_RHSIL, ((size_t)mi * N + r) * 17 + at(17, sub + 4 * u));
    }
};
// y_i = band row i (half width K, four lanes, coefficients b) times x, zero
// for i < nzero; every lane of the four gets the sum
template <int K, class B>
__device__ __forceinline__ cd band_row(const B (&b)[(2 * K + 4) / 4], const cd *x, int i, int N, int nzero)
{
    constexpr int W = 2 * K + 1;
    const int sub = threadIdx.x & 3;
    cd s = mk(0.0, 0.0);
#pragma unroll
    for (int u = 0; u < (W + 3) / 4; u++) {
        const int d = sub + 4 * u, j = i - K + d;
        if (i >= nzero && i < N && d < W && j >= 0 && j < N) s = cadd(s, mmul(b[u], lds_load(x, j)));
    }
    s.x += xor_lane_d<1>(s.x);
    s.y += xor_lane_d<1>(s.y);
    s.x += xor_lane_d<2>(s.x);
    s.y += xor_lane_d<2>(s.y);
    return s;
}

// The transforms behind the psi solve in registers (L = 64 P), one wave each,
// to Z[tr][L] in natural order: tr 0 the odd extension of k w_k and tr 1 the
// even extension of k^2 w_k of the psi coefficients w (its derivatives), tr 2
// w itself, tr 3 and 4 the coefficients of T and xi (null: skipped); and the
// k^2 sums of the derivatives at the two walls, by the half-waves counted
// from the last wave, to Z[5 L ..].  No trailing barrier.
__device__ __forceinline__ void mphase_transforms(const PzDev &p, int P, const cd *w, const cd *cT,
                                                  const cd *cX, const double *cosT, const double *sinT, cd *Z)
{
    const int N = p.N, L = p.L;
    auto in_at = [=](int tr, int j) __attribute__((always_inline)) {
        const int k = j < N ? j : L - j;
        cd y = mk(0.0, 0.0);
        if (tr >= 2) {
            y = lds_load(tr == 2 ? w : tr == 3 ? (cT ? cT : cX) : cX, k);
        } else if (k != 0 && k != N - 1) {
            const cd c = lds_load(w, k);
            const double sc = tr == 0 ? (j < N ? (double)k : -(double)k) : (double)k * (double)k;
            y = mk(sc * c.x, sc * c.y);
        }
        return y;
    };
    // without T, xi's transform takes slot 4 and slot 3 repeats it
    fft_wave_p(
        P, cX ? 5 : cT ? 4 : 3, in_at, [=](int tr, int k, cd z) __attribute__((always_inline)) { lds_store(Z, tr * L + k, z); },
        [=](int q) __attribute__((always_inline)) { return mk(cosT[q], -sinT[q]); });
    const int seg = (int)((blockDim.x - 1 - threadIdx.x) >> 5), hl = threadIdx.x & 31;
    if (seg < 2) {
        double ax = 0, ay = 0, bx = 0, by = 0;
        for (int k = 1 + hl; k <= N - 1; k += 32) {
            const cd wk = lds_load(w, k);
            const double e = k == N - 1 ? 0.5 : 1.0, k2 = (double)k * k;
            const double s1 = seg == 0 || (k & 1) ? e * k2 : -e * k2, s2 = seg == 0 || !(k & 1) ? e * k2 * (k2 - 1.0) : -e * k2 * (k2 - 1.0);
            ax += s1 * wk.x;
            ay += s1 * wk.y;
            bx += s2 * wk.x;
            by += s2 * wk.y;
        }
        for (int o = 16; o > 0; o >>= 1) {
            ax += __shfl_xor(ax, o, 32);
            ay += __shfl_xor(ay, o, 32);
            bx += __shfl_xor(bx, o, 32);
            by += __shfl_xor(by, o, 32);
        }
        if (hl == 0) {
            const double sc = p.icheb_fac / (double)(N - 1);
            lds_store(Z, 5 * L + 2 * seg, mk(ax * sc, ay * sc));
            lds_store(Z, 5 * L + 2 * seg + 1, mk((1.0 / 3.0) * bx * sc, (1.0 / 3.0) * by * sc));
        }
    }
}
// psi and its two radial derivatives at grid point j from those transforms
__device__ __forceinline__ void mphase_psi_at(const PzDev &p, const RadView &R, const cd *Z, const cd *bnd, const cd *w, int j,
                                              cd &ps, cd &dps, cd &d2ps)
{
    const int N = p.N, L = p.L;
    cd d1, d2;
    if (j == 0 || j == N - 1) {
        const int seg = j == 0 ? 0 : 1;
        d1 = lds_load(bnd, 2 * seg);
        d2 = lds_load(bnd, 2 * seg + 1);
    } else {
        const cd zv = lds_load(Z, j), zu = lds_load(Z, L + j);
        dr_bulk(p, R, lds_load(w, N - 1), j, true, -0.5 * zv.y, 0.5 * zv.x, 0.5 * zu.x, 0.5 * zu.y, d1, d2);
    }
    const double a = R.drx(j), b = R.ddrx(j), cf = p.cheb_fac;
    const cd z = lds_load(Z, 2 * L + j);
    ps = mk(cf * z.x, cf * z.y);
    dps = mk(a * d1.x, a * d1.y);
    d2ps = mk(b * d1.x + a * a * d2.x, b * d1.y + a * a * d2.y);
}

// One stage of the m-loop for one azimuthal wavenumber per workgroup:
// finish_explicit_assembly (mloop.f90:169-229) when exp_calc, then
// update_temp_int / update_xi_int (update_temp_integ.f90:179-298) and
// update_psi_int_smat (update_psi_integ_smat.f90:247-573).
//
// What bounds it is the chain of phases of one workgroup (one per mode, 129
// on 256 CUs), each a load or LDS round trip and a barrier.  So the linear
// maps that all modes share are applied as dense products with composed
// matrices (T_M, P_M, P_G, set up in long double): dealiased transform, radial
// derivative of the advective flux, second transform and band of the
// explicit assembly in one product instead of five phases, and transform,
// buoyancy, transform and band of the implicit buoyancy in one instead of
// four.  The barriers order LDS only, the inverses are loaded into registers
// behind the inputs, long before their use, the slots of a multistep scheme
// rotate from the values the right-hand side reads, and everything behind
// the psi solve (up to five transforms, six bands) is one phase.  Measured at
// n_r 97, 129 modes, both scalars: 31.9 us a launch (42.7 us before).
template <int PFS, int PFP, int U>
__device__ __forceinline__ void mphase_body(const PzDev &p, int mi, int istage, int exp_calc)
{
    extern __shared__ double smem[];
    const int N = p.N, m = mi * p.minc;
    const size_t F = (size_t)p.nm * N, off = (size_t)mi * N;
    const int is = istage - 1;
    const PzScheme *ss = p.ss;
    const int tid = threadIdx.x;
    const MpLayout lay(N);
    char *lb = (char *)smem;
    cd *V = (cd *)(lb + lay.vec);
    // e and a of a field are adjacent: the 2 n_r inputs of its explicit assembly
    cd *eT = V, *aT = V + N, *eX = V + 2 * N, *aX = V + 3 * N, *eP = V + 4 * N, *aP = V + 5 * N;
    cd *cT = V + 6 * N, *cX = V + 7 * N, *cP = V + 8 * N;
    cd *psiv = V + 9 * N, *omv = V + 10 * N, *upv = V + 11 * N, *usv = V + 12 * N;
    cd *Tv = V + 13 * N, *Xv = V + 14 * N, *bv = V + 15 * N, *b2 = V + 16 * N, *wv = V + 17 * N;
    cd *PT = V + 18 * N, *QT = V + 19 * N, *PX = V + 20 * N, *QX = V + 21 * N, *PP = V + 22 * N, *QP = V + 23 * N;
    double *cosT = (double *)(lb + lay.cosT), *sinT = (double *)(lb + lay.sinT);
    const bool hT = p.l_heat, hX = p.l_chem;
    cd *red = (cd *)(lb + lay.red), *fbuf = red;
    const int ldi = p.ldi;
    const RadView R((const double *)(lb + lay.rad), N);

    // ---------------- global inputs of this m in one phase ----------------
    // the tables, the explicit-assembly inputs (or the current explicit slot)
    // and the slots of the right-hand sides: three groups of N threads (T, xi,
    // psi), the velocity fields spread over them; every load of a thread is
    // issued before the first is stored
    const int ntab = 2 * p.L + PZ_NRADC * N;
    TableStage tab;
    tab.load(p.cosT, ntab);
    // shared-matrix products: thread groups (one half of the threads for T and
    // xi, the other for psi)
    const int ldm = (N + 3) & ~3, RU = ldm >> 2, half = blockDim.x >> 1, side = tid >= half, ht = tid - side * half;
    const int CG = shared_groups(N, half), cg = ht / RU, ru = ht - cg * RU;
    const double *ME = side ? (m == 0 ? p.P_M0 : p.P_M) : p.T_M;
    const int nME = side && m == 0 ? N : 2 * N;
    SharedMv<U> mv;
    for (int t = tid; t < 3 * N; t += blockDim.x) {
        const int g = t / N, k = t - g * N;
        const size_t q = off + k, qe = is * F + q;
        const bool have = g == 0 ? hT : g == 1 ? hX : true;
        cd *old = g == 0 ? p.T_old : g == 1 ? p.X_old : p.P_old, *impl = g == 0 ? p.T_impl : g == 1 ? p.X_impl : p.P_impl;
        cd *expl = g == 0 ? p.T_expl : g == 1 ? p.X_expl : p.P_expl;
        const cd *dV = g == 0 ? p.dVsT : g == 1 ? p.dVsXi : p.dVsOm;
        cd e = mk(0.0, 0.0), a = e, u1 = e, u2 = e, wall = e, b, c;
        ImexSlots sl;
        if (g < 2 && k < 2) wall = gld(g == 0 ? (k == 0 ? p.topt : p.bott) : (k == 0 ? p.topxi : p.botxi), mi);
        if (have) {
            e = gld(expl, qe);
            sl.load(p, istage, old, impl, expl, q);
        }
        if (exp_calc) {
            if (have) a = gld(dV, q);
            u1 = gld(g == 0 ? p.psi : g == 1 ? p.om : p.up, q);
            if (g == 0) u2 = gld(p.us, q);
            else if (!p.l_buo_imp && (g == 1 ? hT : hX)) u2 = gld(g == 1 ? p.temp : p.xi, q);
        }
        if (t == tid) {
            if (exp_calc && cg < CG) mv.load(ME, ldm, nME, cg, ru, CG);
            tab.store(p.cosT, cosT, ntab);
        }
        if (have) {
            lds_store(g == 0 ? eT : g == 1 ? eX : eP, k, e);
            sl.sum(p, ss, istage, old, impl, expl, q, b, c);
            if (g < 2 && k < 2) b = wall; // tau rows: the boundary value alone
            lds_store(g == 0 ? PT : g == 1 ? PX : PP, k, b);
            lds_store(g == 0 ? QT : g == 1 ? QX : QP, k, c);
        }
        if (exp_calc) {
            lds_store(g == 0 ? aT : g == 1 ? aX : aP, k, a);
            lds_store(g == 0 ? psiv : g == 1 ? omv : upv, k, u1);
            lds_store(g == 0 ? usv : g == 1 ? Tv : Xv, k, u2);
        }
    }
    if (tid >= 3 * N) {
        if (exp_calc && cg < CG) mv.load(ME, ldm, nME, cg, ru, CG);
        tab.store(p.cosT, cosT, ntab);
    }
    const double wcur = imex_weight(p, ss, istage);
    const VecSet<const double> invS(hT ? p.T_inv + off * ldi : p.X_inv + off * ldi, p.X_inv + off * ldi);
    const VecSet<const cd> invP(p.P_inv + off * ldi);
    // the groups above wrote vectors that other threads read next, with or
    // without the explicit part
    lds_barrier();

    // right-hand sides of T and xi at one point
    auto rhsT = [&](int k, cd e) { return k < 2 ? PT[k] : cadd(cadd(PT[k], cscale(wcur, e)), QT[k]); };
    auto rhsX = [&](int k, cd e) { return k < 2 ? PX[k] : cadd(cadd(PX[k], cscale(wcur, e)), QX[k]); };
    // the first columns of the inverses, in flight until their solves
    MatAhead<double, 2, PFS> preS; // T and xi
    MatAhead<cd, 1, PFP> preP;
    // ---------------- explicit assembly -----------------------------------
    if (exp_calc) {
        const double rc2 = p.r_cmb * p.r_cmb;
        for (int t = tid; t < 3 * N; t += blockDim.x) {
            const int g = t / N, k = t - g * N;
            const double rk = R.r(k), h2 = rc2 - rk * rk;
            if (g == 0) {
                if (!hT) continue;
                // finish_exp_temp_int (update_temp_integ.f90:420-438)
                const double s = h2 * R.dtcond(k) + p.tadvz * rk * R.tcond(k);
                eT[k] = csub(cscale(rk, eT[k]), cimul((double)m * s, psiv[k]));
            } else if (g == 1) {
                if (hX) eX[k] = csub(cscale(rk, eX[k]), cimul((double)m * h2 * R.dxicond(k), psiv[k]));
            } else {
                // finish_exp_psi_int_smat (update_psi_integ_smat.f90:832-930)
                cd e = eP[k];
                if (m != 0) {
                    e = cscale(rk, e);
                    if (!p.l_coriolis_imp) e = csub(e, cimul(p.CorFac * (double)m * rk, psiv[k]));
                    if (!p.l_buo_imp) {
                        if (hT) e = csub(e, cimul(p.BuoFac * R.rgrav(k) * (double)m, Tv[k]));
                        if (hX) e = csub(e, cimul(p.ChemFac * R.rgrav(k) * (double)m, Xv[k]));
                    }
                }
                if (p.l_ek_pump) {
                    const double ekp = p.CorFac * R.ekpump(k);
                    if (m == 0) {
                        e = csub(e, cscale(ekp, upv[k]));
                    } else {
                        cd t2 = cadd(omv[k], cscale(R.ekp_up(k), upv[k]));
                        t2 = cadd(t2, cmul(mk(R.ekp_us(k), (double)m * R.ekp_dusdp(k)), usv[k]));
                        e = csub(e, cscale(ekp * rk, t2));
                    }
                }
                eP[k] = e;
            }
        }
        lds_barrier();
        // red: [T][CG][ldm], [xi][CG][ldm], [psi][CG][ldm]
        const int RS = CG * ldm;
        if (cg < CG) {
            if (side) mv.template run<1>(ME, ldm, nME, eP, nullptr, cg, ru, CG, red + 2 * RS);
            else if (hT && hX) mv.template run<2>(ME, ldm, nME, eT, eX, cg, ru, CG, red);
            else if (hT || hX) mv.template run<1>(ME, ldm, nME, hT ? eT : eX, nullptr, cg, ru, CG, red + (hT ? 0 : RS));
        }
        lds_barrier();
        for (int t = tid; t < 3 * N; t += blockDim.x) {
            const int g = t / N, k = t - g * N;
            if ((g == 0 && !hT) || (g == 1 && !hX)) continue;
            const cd e = shared_sum(red + g * RS, CG, ldm, k);
            cd *expl = g == 0 ? p.T_expl : g == 1 ? p.X_expl : p.P_expl;
            expl[is * F + off + k] = e;
            rotate_current(p, expl, off, k, e);
            if (g == 2) eP[k] = e;
            else if (g == 0) aT[k] = rhsT(k, e);
            else aX[k] = rhsX(k, e);
        }
    } else {
        for (int k = tid; k < N; k += blockDim.x) {
            if (hT) {
                rotate_current(p, p.T_expl, off, k, eT[k]);
                aT[k] = rhsT(k, eT[k]);
            }
            if (hX) {
                rotate_current(p, p.X_expl, off, k, eX[k]);
                aX[k] = rhsX(k, eX[k]);
            }
            rotate_current(p, p.P_expl, off, k, eP[k]);
        }
    }
    if (hT && hX) preS.load(N, N, ldi, invS);
    lds_barrier();

    // ---------------- T and xi: bordered solves ----------------------------
    // (update_temp_integ.f90:226-240) by their inverses; implicit buoyancy
    // takes BuoFac T + ChemFac xi from their coefficients (wv)
    const bool buo = p.l_buo_imp && m != 0 && (hT || hX);
    const int CB = shared_groups(N, blockDim.x), cb = tid / RU, rb = tid - cb * RU;
    SharedMv<U> gv;
    auto ahead = [&]() __attribute__((always_inline)) {
        if (buo && cb < CB) gv.load(p.P_G, ldm, N, cb, rb, CB);
        preP.load(N, N, ldi, invP);
    };
    if (hT && hX) {
        preS.apply(N, N, ldi, invS, VecSet<cd>(aT, aX), red, ahead, [&](int k, const cd(&s)[2]) __attribute__((always_inline)) {
            aT[k] = s[0];
            aX[k] = s[1];
            wv[k] = cadd(cscale(p.BuoFac, s[0]), cscale(p.ChemFac, s[1]));
        });
    } else {
        if (hT || hX) block_matvec<double, 1>(N, ldi, invS, VecSet<cd>(hT ? aT : aX), VecSet<cd>(hT ? aT : aX), red);
        ahead();
        for (int k = tid; k < N; k += blockDim.x) wv[k] = hT ? cscale(p.BuoFac, aT[k]) : cscale(p.ChemFac, aX[k]);
    }
    lds_barrier();
    const int inext = (istage == p.nstages) ? 1 : istage + 1;
    // implicit terms for the next stage; also before a CNAB2 start-up step
    // of a multistep scheme, which recomputes them (step_time.f90:417-503)
    const int bridge_next = p.bridge && ss->n_steps + 1 <= p.nold - 1;
    const int lcalc = p.l_imp_calc_rhs[inext - 1] || bridge_next;

    // ---------------- psi -------------------------------------------------
    const double wl = ss->wimp_lin[0];
    if (buo) {
        // implicit buoyancy: RHSE2 costf(-rgrav / r i m (BuoFac T + ChemFac xi))
        if (cb < CB) gv.template run<1>(p.P_G, ldm, N, wv, nullptr, cb, rb, CB, red);
        lds_barrier();
    }
    for (int k = tid; k < N; k += blockDim.x) {
        cd r = cadd(cadd(PP[k], cscale(wcur, eP[k])), QP[k]);
        if (buo) {
            const cd b = cimul((double)m, shared_sum(red, CB, ldm, k));
            b2[k] = b;
            r = cadd(r, cscale(wl, b));
        } else {
            b2[k] = mk(0.0, 0.0);
        }
        aP[k] = r;
    }
    lds_barrier();
    // bordered solve of psi (update_psi_integ_smat.f90:417-432) by its inverse
    preP.apply(N, N, ldi, invP, VecSet<cd>(aP), red, []() {},
               [&](int k, const cd(&s)[1]) __attribute__((always_inline)) { aP[k] = s[0]; });
    lds_barrier();
    const double rc2 = p.r_cmb * p.r_cmb;
    const int Pw = wave_fft_p(p);
    // the bands of the implicit terms go by blocks of 16 rows, four lanes a
    // row: where the transforms run in registers, two blocks to each wave
    // without a transform, the others to the rest behind theirs
    BandRow br;
    const int wave = tid >> 6, nw = blockDim.x >> 6, ntr = m != 0 && Pw ? 3 + (hX ? 2 : hT ? 1 : 0) : nw;
    const int nfree = max(0, nw - ntr), nblk = (N + 15) >> 4, first = min(nblk, 2 * nfree);
    const bool isfree = wave >= ntr;
    const int blk0 = isfree ? wave - ntr : first + wave, dblk = isfree ? nfree : nw - nfree, blk1 = isfree ? first : nblk;
    const int il = (tid & 63) >> 2;
    if (m != 0) br.load(p, mi, blk0 < blk1 ? 16 * blk0 + il : N);
    if (m == 0) {
        // u_phi: omega from the coefficients' derivative (dcheb), grid values
        if (tid < 128) dcheb_waves(p, aP, cP);
        for (int k = tid; k < N; k += blockDim.x) wv[k] = mk(aP[k].x, 0.0); // = costf(real(u_phi)), costf being its own inverse
        lds_barrier();
        if (Pw) {
            VecSet<const cd> din(cP, wv);
            VecSet<cd> dout(omv, upv);
            if (hT) { din.push(aT); dout.push(Tv); }
            if (hX) { din.push(aX); dout.push(Xv); }
            dct_fft(p, din, dout, din.n, 0, cosT, sinT, fbuf);
        } else {
            dct_fft(p, VecSet<const cd>(cP, wv), VecSet<cd>(omv, upv), 2, 0, cosT, sinT, fbuf);
            lds_barrier();
            VecSet<const cd> din;
            VecSet<cd> dout;
            if (hT) { din.push(aT); dout.push(Tv); }
            if (hX) { din.push(aX); dout.push(Xv); }
            if (din.n) dct_fft(p, din, dout, din.n, 0, cosT, sinT, fbuf);
        }
    } else if (Pw) {
        // derivatives and grid values of psi, grid values of T and xi
        mphase_transforms(p, Pw, aP, hT ? aT : nullptr, hX ? aX : nullptr, cosT, sinT, fbuf);
    } else {
        dr_fft(p, R, VecSet<const cd>(aP), VecSet<cd>(cP), VecSet<cd>(bv), 1, cosT, sinT, fbuf, psiv);
        lds_barrier();
        VecSet<const cd> din;
        VecSet<cd> dout;
        if (hT) { din.push(aT); dout.push(Tv); }
        if (hX) { din.push(aX); dout.push(Xv); }
        if (din.n) dct_fft(p, din, dout, din.n, 0, cosT, sinT, fbuf);
    }
    // get_temp_rhs_imp_int (update_temp_integ.f90:471-536) and
    // get_psi_rhs_imp_int_smat (update_psi_integ_smat.f90:960-1115)
    if (m == 0) {
        if (inext == 1) {
            if (hT) bandmv<4>(p, p.T_RHSE2, aT, p.T_old + off, 2);
            if (hX) bandmv<4>(p, p.T_RHSE2, aX, p.X_old + off, 2);
            bandmv<4>(p, p.P_RHSI + (size_t)mi * N * 17, wv, p.P_old + off, 2);
        }
        if (lcalc) {
            if (hT) bandmv<2>(p, p.T_RHSI + (size_t)mi * N * 5, aT, cT, 2);
            if (hX) bandmv<2>(p, p.T_RHSI + (size_t)mi * N * 5, aX, cX, 2);
            bandmv_c<2>(p, p.P_RHSIL + (size_t)mi * N * 17, wv, QP, 2);
        }
    } else {
        for (int bk = blk0; bk < blk1; bk += dblk) {
            const int i = 16 * bk + il;
            if (bk != blk0) br.load(p, mi, i);
            const bool w = (tid & 3) == 0 && i < N;
            if (inext == 1) {
                if (hT) { const cd y = band_row<4>(br.e2, aT, i, N, 2); if (w) p.T_old[off + i] = y; }
                if (hX) { const cd y = band_row<4>(br.e2, aX, i, N, 2); if (w) p.X_old[off + i] = y; }
                const cd y = band_row<8>(br.pi, aP, i, N, 4);
                if (w) p.P_old[off + i] = y;
            }
            if (lcalc) {
                if (hT) { const cd y = band_row<2>(br.ti, aT, i, N, 2); if (w) lds_store(cT, i, y); }
                if (hX) { const cd y = band_row<2>(br.ti, aX, i, N, 2); if (w) lds_store(cX, i, y); }
                const cd y = band_row<8>(br.pl, aP, i, N, 4);
                if (w) lds_store(QP, i, y);
            }
        }
    }
    lds_barrier();
    const cd *Z = fbuf; // mphase_transforms' outputs
    const int L = p.L;
    for (int k = tid; k < N; k += blockDim.x) {
        if (m != 0) {
            cd ps, dps, d2ps;
            if (Pw) {
                mphase_psi_at(p, R, Z, fbuf + 5 * (size_t)L, aP, k, ps, dps, d2ps);
            } else {
                ps = psiv[k];
                dps = cP[k];
                d2ps = bv[k];
            }
            const double rk = R.r(k), h2 = rc2 - rk * rk, or1 = R.or1(k);
            if (bridge_next) psiv[k] = ps;
            p.psi_hat[off + k] = aP[k];
            p.psi[off + k] = ps;
            p.us[off + k] = cimul((double)m * or1 * h2, ps);
            p.up[off + k] = cadd(cscale(-h2, dps), cscale(3.0 * rk, ps));
            const cd o = csub(cscale(-h2, d2ps), cscale(rc2 * or1 - 6.0 * rk, dps));
            p.om[off + k] = cadd(o, cscale(6.0 + (double)m * (double)m * R.or2(k) * h2, ps));
        }
        if (m == 0) {
            const double u0 = upv[k].x, om0 = R.drx(k) * omv[k].x;
            p.us[off + k] = mk(0, 0);
            p.up[off + k] = mk(u0, 0.0);
            p.om[off + k] = mk(om0 + R.or1(k) * u0, 0.0);
        }
        const double cf = p.cheb_fac;
        if (hT) {
            const cd T = m != 0 && Pw ? cscale(cf, Z[3 * (size_t)L + k]) : Tv[k];
            if (bridge_next) Tv[k] = T;
            p.temp_hat[off + k] = aT[k];
            p.temp[off + k] = T;
            if (lcalc) p.T_impl[(inext - 1) * F + off + k] = cscale(p.TdiffFac * p.hdifT[mi], cT[k]);
        }
        if (hX) {
            const cd X = m != 0 && Pw ? cscale(cf, Z[4 * (size_t)L + k]) : Xv[k];
            p.xi_hat[off + k] = aX[k];
            p.xi[off + k] = X;
            if (lcalc) p.X_impl[(inext - 1) * F + off + k] = cscale(p.XidiffFac * p.hdifXi[mi], cX[k]);
        }
    }
    if (!lcalc) return;
    cd *bimp = b2;
    if (bridge_next && p.l_buo_imp && hX && m != 0) {
        // the start-up recomputation passes psi in the composition slot
        // (step_time.f90:475-478): buoyancy of (T, psi) instead of (T, xi)
        lds_barrier();
        for (int k = tid; k < N; k += blockDim.x)
            bv[k] = buoyancy(p, R, m, k, hT ? Tv[k] : mk(0, 0), psiv[k]);
        lds_barrier();
        dct_fft(p, VecSet<const cd>(bv), VecSet<cd>(PT), 1, 0, cosT, sinT, fbuf);
        lds_barrier();
        bandmv<8>(p, p.P_RHSE2, PT, PX, 4);
        bimp = PX;
        lds_barrier();
    }
    for (int k = tid; k < N; k += blockDim.x) {
        cd v = QP[k];
        if (p.l_buo_imp && m != 0) v = cadd(v, bimp[k]);
        p.P_impl[(inext - 1) * F + off + k] = v;
    }
}

// the descriptor is read through a pointer (scalar loads): a by-value copy
// of this size would be materialised in scratch memory
__global__ void __launch_bounds__(PZ_MPHASE_THREADS) k_mphase(const PzDev *__restrict__ pd, int istage, int exp_calc)
{
    mphase_body<10, 16, 8>(*pd, blockIdx.x, istage, exp_calc);
}
__global__ void __launch_bounds__(PZ_MPHASE_THREADS) k_mphase_batch(PzBatch b, int istage, int exp_calc)
{
    const int2 e = b.map[blockIdx.x];
    mphase_body<10, 16, 8>(*b.runs[e.x], e.y, istage, exp_calc);
}
// n_r <= 65 (256 threads): fewer columns ahead and 168 registers, so that
// three workgroups of many small runs share a CU (48 runs at n_r 33: 179 us a
// step, 199 us with the larger form); the sums are the same
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) k_mphase_batch_small(PzBatch b, int istage, int exp_calc)
{
    const int2 e = b.map[blockIdx.x];
    mphase_body<2, 4, 3>(*b.runs[e.x], e.y, istage, exp_calc);
}

// get_start_fields, fresh start of the integration method
// (init_fields.f90:186-255): dT/dr, omega, hats and the first implicit state.
__global__ void __launch_bounds__(256) k_start(const PzDev p __attribute__((grid_constant)))
{
    extern __shared__ double smem[];
    const int mi = blockIdx.x, N = p.N, m = p.idx2m[mi];
    const size_t F = (size_t)p.nm * N, off = (size_t)mi * N;
    (void)F;
    const int tid = threadIdx.x;
    cd *V = (cd *)smem;
    cd *Tv = V, *Xv = V + N, *upv = V + 2 * N, *usv = V + 3 * N, *psv = V + 4 * N;
    cd *cT = V + 5 * N, *cX = V + 6 * N, *cU = V + 7 * N, *cPs = V + 8 * N;
    cd *dT = V + 9 * N, *dU = V + 10 * N, *bv = V + 11 * N, *wv = V + 12 * N, *b2 = V + 13 * N, *t1 = V + 14 * N;
    const bool hT = p.l_heat, hX = p.l_chem;
    for (int k = tid; k < N; k += blockDim.x) {
        Tv[k] = hT ? p.temp[off + k] : mk(0, 0);
        Xv[k] = hX ? p.xi[off + k] : mk(0, 0);
        upv[k] = p.up[off + k];
        usv[k] = p.us[off + k];
        psv[k] = p.psi[off + k];
    }
    __syncthreads();
    {
        VecSet<const cd> din(Tv, Xv, upv, psv);
        VecSet<cd> dout(cT, cX, cU, cPs);
        dct_many(p, din, dout, 4, 0);
    }
    __syncthreads();
    {
        VecSet<const cd> c2(cT, cU);
        VecSet<cd> d2(dT, dU);
        dr_many(p, RadView(p.radc, p.N), c2, d2, VecSet<cd>(), 2);
    }
    __syncthreads();
    for (int k = tid; k < N; k += blockDim.x) {
        if (hT) { p.dtemp[off + k] = dT[k]; p.temp_hat[off + k] = cT[k]; }
        if (hX) p.xi_hat[off + k] = cX[k];
        p.psi_hat[off + k] = cPs[k];
        cd o = cadd(dU[k], cscale(p.or1[k], upv[k]));
        p.om[off + k] = csub(o, cmul(mk(0.0, p.or1[k] * (double)m), usv[k]));
    }
    // scalar implicit states (istage = 1, l_calc_lin = .true.)
    if (hT) {
        bandmv<4>(p, p.T_RHSE2, cT, p.T_old + off, 2);
        bandmv<2>(p, p.T_RHSI + (size_t)mi * N * 5, cT, t1, 2);
        __syncthreads();
        for (int k = tid; k < N; k += blockDim.x) p.T_impl[off + k] = cscale(p.TdiffFac * p.hdifT[mi], t1[k]);
        __syncthreads();
    }
    if (hX) {
        bandmv<4>(p, p.T_RHSE2, cX, p.X_old + off, 2);
        bandmv<2>(p, p.T_RHSI + (size_t)mi * N * 5, cX, t1, 2);
        __syncthreads();
        for (int k = tid; k < N; k += blockDim.x) p.X_impl[off + k] = cscale(p.XidiffFac * p.hdifXi[mi], t1[k]);
        __syncthreads();
    }
    // psi: the reference passes psi in the composition slot (init_fields.f90:250-251)
    if (m == 0) {
        // work_r = costf(real(up(m=0)))
        for (int k = tid; k < N; k += blockDim.x) bv[k] = mk(upv[k].x, 0.0);
        __syncthreads();
        VecSet<const cd> di(bv);
        VecSet<cd> dd(wv);
        dct_many(p, di, dd, 1, 0);
        __syncthreads();
        for (int k = tid; k < N; k += blockDim.x) wv[k] = mk(wv[k].x, 0.0);
        __syncthreads();
        bandmv<4>(p, p.P_RHSI + (size_t)mi * N * 17, wv, p.P_old + off, 2);
        bandmv_c<2>(p, p.P_RHSIL + (size_t)mi * N * 17, wv, p.P_impl + off, 2);
    } else {
        bandmv<8>(p, p.P_RHSI + (size_t)mi * N * 17, cPs, p.P_old + off, 4);
        bandmv_c<8>(p, p.P_RHSIL + (size_t)mi * N * 17, cPs, t1, 4);
        if (p.l_buo_imp) {
            for (int k = tid; k < N; k += blockDim.x) bv[k] = buoyancy(p, RadView(p.radc, p.N), m, k, Tv[k], psv[k]);
            __syncthreads();
            VecSet<const cd> di(bv);
            VecSet<cd> dd(wv);
            dct_many(p, di, dd, 1, 0);
            __syncthreads();
            bandmv<8>(p, p.P_RHSE2, wv, b2, 4);
        }
        __syncthreads();
        for (int k = tid; k < N; k += blockDim.x) {
            cd v = t1[k];
            if (p.l_buo_imp) v = cadd(v, b2[k]);
            p.P_impl[off + k] = v;
        }
    }
}

// radial profiles for the kinetic energies (outputs.f90:458-467): per r,
// sum over m of cc2real(us), cc2real(up) and the m = 0 part of up
__global__ void k_ekin_profiles(const PzDev p __attribute__((grid_constant)), double *out)
{
    const int nr = blockIdx.x * blockDim.x + threadIdx.x;
    if (nr >= p.N) return;
    double us2 = 0.0, up2 = 0.0, upa = 0.0;
    for (int i = 0; i < p.nm; i++) {
        const int m = p.idx2m[i];
        cd u = p.us[(size_t)i * p.N + nr], v = p.up[(size_t)i * p.N + nr];
        double a = m == 0 ? u.x * u.x : 2.0 * (u.x * u.x + u.y * u.y);
        double b = m == 0 ? v.x * v.x : 2.0 * (v.x * v.x + v.y * v.y);
        us2 += a;
        up2 += b;
        if (m == 0) upa += b;
    }
    out[nr] = us2;
    out[p.N + nr] = up2;
    out[2 * p.N + nr] = upa;
}

// ---- unit-operator kernels on [vec][n_r] device arrays ----
__global__ void __launch_bounds__(256) k_costf_vecs(const PzDev p __attribute__((grid_constant)), cd *f)
{
    extern __shared__ double smem[];
    cd *a = (cd *)smem, *b = a + p.N, *buf = b + p.N;
    cd *x = f + (size_t)blockIdx.x * p.N;
    for (int k = threadIdx.x; k < p.N; k += blockDim.x) a[k] = x[k];
    __syncthreads();
    VecSet<const cd> din(a);
    VecSet<cd> dout(b);
    dct_fft(p, din, dout, 1, 0, p.cosT, p.sinT, buf);
    __syncthreads();
    for (int k = threadIdx.x; k < p.N; k += blockDim.x) x[k] = b[k];
}

__global__ void __launch_bounds__(256) k_dr_vecs(const PzDev p __attribute__((grid_constant)), const cd *f, cd *df, cd *ddf, int l_dct_in)
{
    extern __shared__ double smem[];
    cd *a = (cd *)smem, *c = a + p.N, *d1 = c + p.N, *d2 = d1 + p.N, *buf = d2 + p.N;
    const size_t off = (size_t)blockIdx.x * p.N;
    for (int k = threadIdx.x; k < p.N; k += blockDim.x) a[k] = f[off + k];
    __syncthreads();
    if (l_dct_in) {
        VecSet<const cd> din(a);
        VecSet<cd> dout(c);
        dct_fft(p, din, dout, 1, 0, p.cosT, p.sinT, buf);
    } else {
        for (int k = threadIdx.x; k < p.N; k += blockDim.x) c[k] = a[k];
    }
    __syncthreads();
    VecSet<const cd> cc(c);
    VecSet<cd> o1(d1), o2(d2);
    dr_fft(p, RadView(p.radc, p.N), cc, o1, ddf ? o2 : VecSet<cd>(), 1, p.cosT, p.sinT, buf);
    __syncthreads();
    for (int k = threadIdx.x; k < p.N; k += blockDim.x) {
        df[off + k] = d1[k];
        if (ddf) ddf[off + k] = d2[k];
    }
}

// get_dr / get_ddr of n_m columns in the reference's layout f(n_m, n_r), m
// fastest: a workgroup reads its V columns (V n_r values, runs of V), transforms
// them in LDS as k_dr_vecs does, and writes them back in the same layout, so
// that f and df may be the same array.  One launch and two passes over memory
// in place of the layout change, transform and two layout changes of the
// staged form: 4.3 us a call at n_r 33 with 33 columns (13.6 us), 25.9 us at
// n_r 193 with 1358 (26.4 us; the long Stockham stages bound it).  More columns a workgroup fill its
// threads (48 butterflies a stage and column at n_r 193) and lengthen the runs;
// consecutive tiles share a chiplet, whose L2 then holds their common lines.
__host__ __device__ inline size_t dr_ref_lds(int N, int V)
{
    const size_t L = 2 * (size_t)N - 2;
    return (4 * (size_t)V * N + 4 * V * L + 4 * V + 16) * sizeof(cd);
}
// columns a workgroup: as many as leave two workgroups for every CU's worth of
// LDS (80 KB each) and the chip's 256 CUs at least one
inline int dr_ref_vectors(int N, int n_m)
{
    for (int V = 4; V > 1; V >>= 1)
        if (dr_ref_lds(N, V) <= 80 * 1024 && n_m >= 256 * V) return V;
    return 1;
}
__global__ void __launch_bounds__(256) k_dr_ref(const PzDev *__restrict__ pd, const cd *f, cd *df, cd *ddf, int n_m, int l_dct_in, int V)
{
    extern __shared__ double smem[];
    const PzDev &p = *pd;
    const int N = p.N, tiles = (n_m + V - 1) / V, per = (tiles + 7) >> 3;
    const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (tile >= tiles) return;
    const int m0 = tile * V, nv = min(V, n_m - m0), sh = V == 4 ? 2 : V - 1; // V is 1, 2 or 4
    cd *a = (cd *)smem, *c = a + V * N, *d1 = c + V * N, *d2 = d1 + V * N, *buf = d2 + V * N;
    for (int t = threadIdx.x; t < V * N; t += blockDim.x) {
        const int k = t >> sh, v = t & (V - 1);
        lds_store(a, v * N + k, v < nv ? gld(f, (size_t)k * n_m + m0 + v) : mk(0.0, 0.0));
    }
    lds_barrier();
    VecSet<const cd> in, cc;
    VecSet<cd> co, o1, o2;
    for (int v = 0; v < V; v++) {
        in.push(a + v * N);
        co.push(c + v * N);
        cc.push(l_dct_in ? c + v * N : a + v * N);
        o1.push(d1 + v * N);
        if (ddf) o2.push(d2 + v * N);
    }
    if (l_dct_in) {
        dct_fft(p, in, co, V, 0, p.cosT, p.sinT, buf);
        lds_barrier();
    }
    dr_fft(p, RadView(p.radc, N), cc, o1, o2, V, p.cosT, p.sinT, buf);
    lds_barrier();
    for (int t = threadIdx.x; t < V * N; t += blockDim.x) {
        const int k = t >> sh, v = t & (V - 1);
        if (v >= nv) continue;
        const size_t q = (size_t)k * n_m + m0 + v;
        df[q] = lds_load(d1, v * N + k);
        if (ddf) ddf[q] = lds_load(d2, v * N + k);
    }
}

// azimuthal transforms, one radius per block: grid real [rad][n_phi],
// spectral [rad][nm]
__global__ void __launch_bounds__(256) k_phi_fft(const PzDev p __attribute__((grid_constant)), const double *grid, cd *spec)
{
    extern __shared__ double smem[];
    const int n = p.nphi, nm = p.nm;
    cd *a = (cd *)smem, *b = a + n;
    const double *g = grid + (size_t)blockIdx.x * n;
    for (int j = threadIdx.x; j < n; j += blockDim.x) a[j] = mk(g[j], 0.0);
    __syncthreads();
    cd *Z = fft_lds(p, a, b, n, 1, -1);
    for (int i = threadIdx.x; i < nm; i += blockDim.x) spec[(size_t)blockIdx.x * nm + i] = cdivr(Z[i], (double)n);
}

__global__ void __launch_bounds__(256) k_phi_ifft(const PzDev p __attribute__((grid_constant)), const cd *spec, double *grid)
{
    extern __shared__ double smem[];
    const int n = p.nphi, nm = p.nm;
    cd *a = (cd *)smem, *b = a + n;
    const cd *s = spec + (size_t)blockIdx.x * nm;
    for (int k = threadIdx.x; k < n; k += blockDim.x) {
        cd z = mk(0, 0);
        if (k == 0) z = mk(s[0].x, 0.0);
        else if (k < nm) z = s[k];
        else if (n - k < nm) z = cconj(s[n - k]);
        a[k] = z;
    }
    __syncthreads();
    cd *Z = fft_lds(p, a, b, n, 1, +1);
    for (int j = threadIdx.x; j < n; j += blockDim.x) grid[(size_t)blockIdx.x * n + j] = Z[j].x;
}
