// sectorq.hip -- persistent work-queue eigensolver for the small sectors of a
// batched solve.
//
// The per-sector work of ed_diag_c (ED_DIAG.f90:115-228) for a sector of
// dimension D is a thick-restart Lanczos with full reorthogonalisation and
// multiplet-completing deflation rounds.  Driven from the host, a sector of a
// few thousand states costs seven launches per Krylov step and a host round
// trip per restart, and the kernels are far too small to fill the chip.  Here one launch
// takes a queue of such sectors (largest first): each 1024-lane workgroup
// pops a sector from an atomic counter and runs the whole solve for it --
// H*v, the three-term steps and classical Gram-Schmidt (one pass for two
// steps), restarts, the Rayleigh-Ritz eigenproblem of the projected matrix
// (parallel cyclic Jacobi on the matrix in LDS), the deflation rounds and the
// explicit residuals -- with the Krylov basis in its own slice of HBM, which
// stays in the XCD's L2 at these sizes.  Workgroups leave when the queue is
// empty; every loop inside is bounded (Krylov steps by the iteration budget,
// Jacobi sweeps, deflation rounds by neig + 1).
//
// The algorithm is the one of trl_run / trl_deflated (krylov.hip): the same
// start vectors, three-term steps, restart rule, convergence test and
// keep/evict rules.  A pair of steps whose norm comes out too small falls back
// to passes of its own here at once (on the host the rest of the cycle is taken again), and
// the eigensolver of the projected matrix differs (Jacobi here, Householder + QL
// on the host), so results agree to the solver tolerance rather than bit for
// bit.
//
// Bound by the gathers of H*v (address by address through L1), the serial
// rounds of Jacobi (0.75 us each) and the latency of L2.  Hence four columns
// on one read of the up hops, eight basis rows in flight, sums of all rows behind one barrier, rotations
// without divisions and two barriers a Jacobi round; every helper is inlined at
// one place, so that the basis pointers stay scalar and the registers of 1024
// lanes suffice.  Per step (18 basis vectors), before -> now: 60 -> 42 us at
// 1,960 states, 93 -> 68 us at 4,900, 260 -> 167 us at 14,400; the batched
// solves of Ns = 8 (two orbitals, all states at once) 99 -> 73 ms and of
// Ns = 10 at finite temperature 132 -> 99 ms.
#include "dmed_internal.h"
#include "tridiag_device.h"
#include "wave_device.h"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <vector>

namespace dmed {

namespace {

constexpr int kQBlock = 1024;      // lanes per workgroup
constexpr int kQMaxM = 64;         // Krylov basis size limit (as trl_run)
constexpr int kQMaxNeig = 16;      // eigenpairs per sector
constexpr int kQMaxRows = kQMaxNeig + kQMaxM;
constexpr int kQWaves = kQBlock / 64;

// One sector of the queue.  Device pointers; the workspace slices are
// disjoint per task.
struct SqTask {
    const int32_t *hu_idx, *hd_idx;
    const double *hu_val, *hd_val;
    const double *du, *dd, *W;
    const uint8_t *impu, *impd;
    int32_t dup, ddw, nhu, nhd, nimp;
    int32_t dim;
    int32_t neig, m, maxit, lowest;
    double tol, degen;
    double *V, *Vs, *w, *Y, *X;         // (m+1)D, (m+1)D, D, neig*D, neig*D
    double **evecs;                     // neig output vectors (ascending energy)
    double *evals, *resid;              // [neig]
    int32_t *info;                      // nout, status, H*v count
};

// ---------------------------------------------------------- block helpers
struct Shared {
    double T[kQMaxM * kQMaxM];          // projected matrix, column-major
    double A[kQMaxM * kQMaxM];          // Jacobi work copy
    double S[kQMaxM * kQMaxM];          // Ritz rotation, column q = vector q
    double c[2 * kQMaxRows + 1];
    double rows[(2 * kQMaxRows + 1) * kQWaves];     // wave sums of wg_dots
    double red[2 * kQWaves];
    double theta[kQMaxM];
    double jc[kQMaxM / 2], js[kQMaxM / 2];
    int order[kQMaxM];
    double th[kQMaxNeig], rr[kQMaxNeig];
    double ke[kQMaxNeig], kr[kQMaxNeig];
    int kslot[kQMaxNeig];
    double bcast;
    int ibcast;
};

// a condition that is the same in every lane, for the compiler to know it
__device__ __forceinline__ bool uniform(bool c) { return __builtin_amdgcn_readfirstlane((int)c) != 0; }

// workgroup sums of a (and b), the same values in every lane: the waves' sums
// meet in LDS and every lane adds them up in order
__device__ __forceinline__ double wg_sum(double a, Shared &sh)
{
    a = wave_sum63(a);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 63) sh.red[w] = a;
    __syncthreads();
    a = 0.0;
#pragma unroll
    for (int k = 0; k < kQWaves; ++k) a += sh.red[k];
    __syncthreads();
    return a;
}

__device__ __forceinline__ void wg_sum2(double &a, double &b, Shared &sh)
{
    a = wave_sum63(a);
    b = wave_sum63(b);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 63) {
        sh.red[w] = a;
        sh.red[kQWaves + w] = b;
    }
    __syncthreads();
    a = b = 0.0;
#pragma unroll
    for (int k = 0; k < kQWaves; ++k) {
        a += sh.red[k];
        b += sh.red[kQWaves + k];
    }
    __syncthreads();
}

// counter-based hash in [-1, 1): the start vectors of krylov.hip
__device__ __forceinline__ double q_hash_uniform(uint64_t seed, uint64_t i)
{
    uint64_t z = seed + 0x9e3779b97f4a7c15ull * (i + 1);
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    z = z ^ (z >> 31);
    return (double)(z >> 11) * (2.0 / 9007199254740992.0) - 1.0;
}

// y = H x over the sector (the tile kernel's per-element sum); returns the
// lane's part of <x, y>.  A lane keeps one row of the D_up x D_dw matrix and
// takes four of its columns at a time: the up hops of the row are read once for
// the four, and the four gathers of a hop are in flight together.  Rows past
// the workgroup's lanes (D_up > 1024) come in further rounds.  Bound by the
// rate of the gathers; more of them in flight (four hops) change nothing.
__device__ __forceinline__ double wg_hxv(const SqTask &t, const double *__restrict__ x, double *__restrict__ y)
{
    const int dup = t.dup, ddw = t.ddw, nhu = t.nhu, nhd = t.nhd;
    const int G = max(1, kQBlock / dup);
    const int g = dup <= kQBlock ? (int)threadIdx.x / dup : 0;
    double s = 0.0;
    if (g < G) {
        for (int iu = threadIdx.x - g * dup; iu < dup; iu += dup <= kQBlock ? dup : kQBlock) {
            const double du = t.du[iu];
            const int bu = t.impu[iu] * t.nimp;
            for (int c0 = g; c0 < ddw; c0 += 4 * G) {
                int id[4], cb[4];
                double xo[4], acc[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    id[r] = min(c0 + r * G, ddw - 1);   // past the last: not stored
                    cb[r] = id[r] * dup;
                    xo[r] = x[cb[r] + iu];
                    acc[r] = (du + t.dd[id[r]] + t.W[bu + t.impd[id[r]]]) * xo[r];
                }
                for (int h = 0; h < nhu; ++h) {
                    const int j = t.hu_idx[h * dup + iu];
                    const double v = t.hu_val[h * dup + iu];
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[r] += v * x[cb[r] + j];
                }
                for (int h = 0; h < nhd; ++h) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int q = h * ddw + id[r];
                        acc[r] += t.hd_val[q] * x[t.hd_idx[q] * dup + iu];
                    }
                }
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (c0 + r * G < ddw) {
                        y[cb[r] + iu] = acc[r];
                        s += xo[r] * acc[r];
                    }
            }
        }
    }
    __syncthreads();
    return s;
}

__device__ __forceinline__ void wg_copy(double *__restrict__ d, const double *__restrict__ s, int n)
{
    for (int e = threadIdx.x; e < n; e += kQBlock) d[e] = s[e];
    __syncthreads();
}

// Projections on the rows Y[0..ny) then V[0..nv) = 0..nr-1.  NV = 1: out[r] =
// <row r, w1>, out[nr] = ||w1||^2.  NV = 2: out[2r] = <row r, w1>, out[2r+1] =
// <row r, w2>, out[2 nr] = <w1, w2>.  Eight rows' loads are in flight
// together; the waves' sums of all rows meet in LDS behind one barrier.
template <int NV>
__device__ __forceinline__ void wg_dots(const double *__restrict__ Y, int ny, const double *__restrict__ V, int nv,
                        const double *__restrict__ w1, const double *__restrict__ w2, int n,
                        double *out, Shared &sh)
{
    const int nr = ny + nv;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    double sw = 0.0;
    for (int e = threadIdx.x; e < n; e += kQBlock) sw += w1[e] * (NV == 1 ? w1[e] : w2[e]);
    for (int r0 = 0; r0 < nr; r0 += 8) {
        const double *b[8];
        double s1[8], s2[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int r = min(r0 + q, nr - 1);
            b[q] = r < ny ? Y + (size_t)r * n : V + (size_t)(r - ny) * n;
            s1[q] = s2[q] = 0.0;
        }
        for (int e = threadIdx.x; e < n; e += kQBlock) {
            const double a1 = w1[e], a2 = NV == 1 ? 0.0 : w2[e];
            double x[8];
#pragma unroll
            for (int q = 0; q < 8; ++q)
                if (r0 + q < nr) x[q] = b[q][e];
#pragma unroll
            for (int q = 0; q < 8; ++q)
                if (r0 + q < nr) {
                    s1[q] += x[q] * a1;
                    if (NV == 2) s2[q] += x[q] * a2;
                }
        }
#pragma unroll
        for (int q = 0; q < 8; ++q)
            if (r0 + q < nr) {
                const double t1 = wave_sum63(s1[q]), t2 = NV == 2 ? wave_sum63(s2[q]) : 0.0;
                if (lane == 63) {
                    sh.rows[NV * (r0 + q) * kQWaves + wv] = t1;
                    if (NV == 2) sh.rows[(2 * (r0 + q) + 1) * kQWaves + wv] = t2;
                }
            }
    }
    sw = wave_sum63(sw);
    if (lane == 63) sh.rows[NV * nr * kQWaves + wv] = sw;
    __syncthreads();
    for (int r = threadIdx.x; r < NV * nr + 1; r += kQBlock) {
        double t = 0.0;
#pragma unroll
        for (int k = 0; k < kQWaves; ++k) t += sh.rows[r * kQWaves + k];
        out[r] = t;
    }
    __syncthreads();
}

// NV = 1: w2 -= sum_r c[r] row_r.  NV = 2, c from wg_dots<2>: w1 becomes
// s (w1 - sum_r c[2r] row_r) and w2 loses sum_r c[2r+1] row_r + s^2 c[2 nr] w1
// (the old w1).  Returns the new ||w2||^2.
template <int NV>
__device__ __forceinline__ double wg_subtract(const double *__restrict__ Y, int ny, const double *__restrict__ V,
                              int nv, double *__restrict__ w1, double *__restrict__ w2, int n,
                              const double *c, double s, Shared &sh)
{
    const int nr = ny + nv;
    double s2 = 0.0;
    for (int e = threadIdx.x; e < n; e += kQBlock) {
        double t1 = 0.0, t2 = 0.0;
        for (int r0 = 0; r0 < nr; r0 += 8) {
            double x[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int r = r0 + q;
                if (r < nr) x[q] = (r < ny ? Y + (size_t)r * n : V + (size_t)(r - ny) * n)[e];
            }
#pragma unroll
            for (int q = 0; q < 8; ++q)
                if (r0 + q < nr) {
                    t2 += x[q] * c[NV * (r0 + q) + NV - 1];
                    if (NV == 2) t1 += x[q] * c[2 * (r0 + q)];
                }
        }
        double r = w2[e] - t2;
        if (NV == 2) {
            const double a = s * w1[e];
            r -= s * c[2 * nr] * a;
            w1[e] = a - s * t1;
        }
        w2[e] = r;
        s2 += r * r;
    }
    return wg_sum(s2, sh);
}

// Classical Gram-Schmidt of w against Y[0..nl) and V[0..jmax), repeated once
// when the first pass cancelled more than half of ||w||^2; the V coefficients
// of both passes are summed into cv[0..jmax).  Returns the final ||w||^2.
__device__ __forceinline__ double wg_orth(const double *Y, int nl, const double *V, int jmax, double *w, int n,
                          double *cv, Shared &sh)
{
    const int rows = nl + jmax;
    double n1 = 0.0;
#pragma unroll 1
    for (int pass = 0; pass < 2; ++pass) {
        wg_dots<1>(Y, nl, V, jmax, w, nullptr, n, sh.c, sh);
        const double n0 = sh.c[rows];
        if (rows <= 0) return n0;
        n1 = wg_subtract<1>(Y, nl, V, jmax, nullptr, w, n, sh.c, 0.0, sh);
        for (int r = threadIdx.x; r < jmax; r += kQBlock)
            cv[r] = pass == 0 ? sh.c[nl + r] : cv[r] + sh.c[nl + r];
        __syncthreads();
        if (!uniform(n1 < 0.5 * n0)) break;
    }
    return n1;
}

// dst = w / sqrt(nrm2) (0 for a zero norm)
__device__ __forceinline__ void wg_normalize(double *dst, const double *w, int n, double nrm2)
{
    const double r = sqrt(nrm2);
    const double a = r > 0.0 ? 1.0 / r : 0.0;
    for (int e = threadIdx.x; e < n; e += kQBlock) dst[e] = a * w[e];
    __syncthreads();
}

// Vs[:, 0..k) = V[:, 0..m) S[0..m, 0..k), eight outputs of two elements a
// pass.  S goes through sh.A (free by now) with the outputs of a row next to
// each other, two to an LDS read.
__device__ __forceinline__ void wg_rotate(const double *__restrict__ V, double *__restrict__ Vs, int n, int m,
                          int k, Shared &sh)
{
    double *A = sh.A;
    for (int q0 = 0; q0 < k; q0 += 8) {
        for (int i = threadIdx.x; i < 8 * m; i += kQBlock) {
            const int j = i >> 3, q = q0 + (i & 7);
            A[i] = q < k ? sh.S[q * m + j] : 0.0;
        }
        __syncthreads();
        for (int e = threadIdx.x; e < n; e += 2 * kQBlock) {
            const int e2 = min(e + kQBlock, n - 1);
            double a1[8], a2[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) a1[q] = a2[q] = 0.0;
#pragma unroll 4
            for (int j = 0; j < m; ++j) {
                const double x1 = V[(size_t)j * n + e], x2 = V[(size_t)j * n + e2];
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    a1[q] += x1 * A[8 * j + q];
                    a2[q] += x2 * A[8 * j + q];
                }
            }
#pragma unroll
            for (int q = 0; q < 8; ++q)
                if (q0 + q < k) {
                    Vs[(size_t)(q0 + q) * n + e] = a1[q];
                    if (e + kQBlock < n) Vs[(size_t)(q0 + q) * n + e2] = a2[q];
                }
        }
        __syncthreads();
    }
}

// Eigen-decomposition of the symmetric m x m matrix sh.A (column-major,
// destroyed): eigenvalues ascending in sh.theta, eigenvectors in the columns
// of sh.S.  Parallel cyclic Jacobi: m/2 disjoint rotations per round in the
// round-robin order, m - 1 rounds per sweep, at most 60 sweeps.
__device__ __forceinline__ void wg_jacobi(int m, Shared &sh)
{
    double *A = sh.A, *S = sh.S;
    for (int e = threadIdx.x; e < m * m; e += kQBlock) S[e] = (e % m == e / m) ? 1.0 : 0.0;
    __syncthreads();
    const int mm = (m + 1) & ~1;           // players, with a dummy when m is odd
    const int np = mm / 2;
    // it/np and it/m for it < 2^12 by a multiplication
    const unsigned inp = (1u << 20) / np + 1, im = (1u << 20) / m + 1;
    for (int sweep = 0; sweep < 60 && m > 1; ++sweep) {
        double off = 0.0, tot = 0.0;
        for (int e = threadIdx.x; e < m * m; e += kQBlock) {
            const double a = A[e];
            if (e % m != e / m) off += a * a;
            tot += a * a;
        }
        wg_sum2(off, tot, sh);
        if (uniform(off <= 1e-32 * tot)) break;
        for (int r = 0; r < mm - 1; ++r) {
            if ((int)threadIdx.x < np) {
                const int k = threadIdx.x;
                int p, q;
                if (k == 0) {
                    p = mm - 1;
                    q = r;
                } else {
                    p = r + k < mm - 1 ? r + k : r + k - (mm - 1);
                    q = r >= k ? r - k : r - k + (mm - 1);
                }
                double c = 1.0, s = 0.0;
                if (p < m && q < m) {
                    const double apq = A[q * m + p];
                    const double app = fabs(A[p * m + p]), aqq = fabs(A[q * m + q]);
                    // a rotation below the diagonals' rounding only zeroes a_pq
                    if (app + 1e3 * fabs(apq) == app && aqq + 1e3 * fabs(apq) == aqq) {
                        A[q * m + p] = 0.0;
                        A[p * m + q] = 0.0;
                    } else if (fabs(apq) > 1e-140) {
                        // cos 2x = |d|/h, sin 2x = b/h, h = sqrt(d^2 + b^2):
                        // c^2 = (1 + cos 2x)/2, s = sin 2x/(2c); no division
                        const double d = A[q * m + q] - A[p * m + p], b = 2.0 * apq;
                        const double ih = rsqrt_series(d * d + b * b);
                        const double c2 = 0.5 + 0.5 * fabs(d) * ih, ic = rsqrt_series(c2);
                        c = c2 * ic;
                        s = 0.5 * (d >= 0.0 ? b : -b) * ih * ic;
                    }
                }
                sh.jc[k] = c;
                sh.js[k] = s;
                sh.order[2 * k] = p;
                sh.order[2 * k + 1] = q;
            }
            __syncthreads();
            // A <- J^T A J: the 2x2 blocks of a row pair and a column pair are
            // independent of each other, columns then rows within a block; the
            // off-diagonal of a rotated pair's own block is zero by
            // construction.  And S <- S J.  An index m (odd m) is the dummy.
            const int nblk = np * np;
            for (int it = threadIdx.x; it < nblk + np * m; it += kQBlock) {
                if (it < nblk) {
                    const int kr = (int)((unsigned)it * inp >> 20), kc = it - kr * np;
                    const int pr = sh.order[2 * kr], qr = sh.order[2 * kr + 1];
                    const int pc = sh.order[2 * kc], qc = sh.order[2 * kc + 1];
                    const double cr = sh.jc[kr], sr = sh.js[kr], cc = sh.jc[kc], sc = sh.js[kc];
                    if (sr == 0.0 && sc == 0.0) continue;
                    const bool vr = pr < m && qr < m, vc = pc < m && qc < m;
                    if (vr && vc) {
                        const double app = A[pc * m + pr], aqp = A[pc * m + qr];
                        const double apq = A[qc * m + pr], aqq = A[qc * m + qr];
                        const double bpp = cc * app - sc * apq, bpq = sc * app + cc * apq;
                        const double bqp = cc * aqp - sc * aqq, bqq = sc * aqp + cc * aqq;
                        const bool own = kr == kc;
                        A[pc * m + pr] = cr * bpp - sr * bqp;
                        A[pc * m + qr] = own ? 0.0 : sr * bpp + cr * bqp;
                        A[qc * m + pr] = own ? 0.0 : cr * bpq - sr * bqq;
                        A[qc * m + qr] = sr * bpq + cr * bqq;
                    } else if (vr) {                // one column, the two rows
                        const int j = pc < m ? pc : qc;
                        const double apj = A[j * m + pr], aqj = A[j * m + qr];
                        A[j * m + pr] = cr * apj - sr * aqj;
                        A[j * m + qr] = sr * apj + cr * aqj;
                    } else if (vc) {                // one row, the two columns
                        const int i = pr < m ? pr : qr;
                        const double aip = A[pc * m + i], aiq = A[qc * m + i];
                        A[pc * m + i] = cc * aip - sc * aiq;
                        A[qc * m + i] = sc * aip + cc * aiq;
                    }
                } else {
                    const int k = (int)((unsigned)(it - nblk) * im >> 20), i = it - nblk - k * m;
                    const int p = sh.order[2 * k], q = sh.order[2 * k + 1];
                    if (p >= m || q >= m || sh.js[k] == 0.0) continue;
                    const double c = sh.jc[k], s = sh.js[k];
                    const double vip = S[p * m + i], viq = S[q * m + i];
                    S[p * m + i] = c * vip - s * viq;
                    S[q * m + i] = s * vip + c * viq;
                }
            }
            __syncthreads();
        }
    }
    // ascending order, equal values in index order: every lane counts those
    // before its own; then the columns of S are permuted through A, which is
    // no longer needed
    const int own = threadIdx.x;
    double d = 0.0;
    if (own < m) {
        d = A[own * m + own];
        sh.order[own] = own;            // stays an index also among NaN
        sh.theta[own] = d;
    }
    __syncthreads();
    if (own < m) {
        int rank = 0;
        for (int i = 0; i < m; ++i) {
            const double v = A[i * m + i];
            rank += i < own ? !(v > d) : v < d;
        }
        sh.order[rank] = own;
        sh.theta[rank] = d;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < m * m; e += kQBlock) A[e] = S[e];
    __syncthreads();
    for (int e = threadIdx.x; e < m * m; e += kQBlock) {
        const int q = e / m, j = e - q * m;
        S[q * m + j] = A[sh.order[q] * m + j];
    }
    __syncthreads();
}

// One thick-restart Lanczos run (trl_run): the `want` lowest eigenpairs of H
// on the complement of Y[0..nl).  Ritz values to sh.th, residual norms to
// sh.rr, Ritz vectors to X.  V and Vs swap roles at every rotation; the
// caller's pointers are updated.  Returns 0 or DMED_ENOCONV.
__device__ __forceinline__ int wg_trl(const SqTask &t, int want, int m, int maxit, double tol, int nl,
                      uint64_t seed, double *&V, double *&Vs, int &used, Shared &sh)
{
    const int n = t.dim;
    const int avail = n - nl;
    m = max(m, want + 2);
    m = min(m, kQMaxM);
    m = min(m, avail);
    const bool full = m == avail;
    double *w = t.w;
    for (int e = threadIdx.x; e < n; e += kQBlock) V[e] = q_hash_uniform(seed, (uint64_t)e);
    for (int e = threadIdx.x; e < m * m; e += kQBlock) sh.T[e] = 0.0;
    __syncthreads();
    int k = 0;
    double beta_last = 0.0, hn = 0.0;      // hn: scale of H, from the coefficients
    bool converged = false, fresh = true;  // fresh: no start vector yet
    for (;;) {
        // step j leaves v_{j+1}; step -1 is the start vector, which only has
        // to be orthogonalised
        for (int j = fresh ? -1 : k; j < m;) {
            const double *vj = V + (size_t)j * n;
            double *w1 = V + (size_t)(j + 1) * n;
            double al = 0.0, be = 0.0, al2 = 0.0, nn = 0.0;
            if (j >= 0) {
                al = wg_hxv(t, vj, w1);
                ++used;
            }
            // step j > k: the three-term step first, w1 -= alpha v_j +
            // beta_{j-1} v_{j-1}
            bool pair = false;
            if (j > k) {
                const double *vjm = vj - n;
                al = wg_sum(al, sh);
                double s2 = 0.0;
                for (int e = threadIdx.x; e < n; e += kQBlock) {
                    const double r = w1[e] - al * vj[e] - beta_last * vjm[e];
                    w1[e] = r;
                    s2 += r * r;
                }
                be = sqrt(wg_sum(s2, sh));
                hn = fmax(hn, fmax(fabs(al), be));
                pair = j + 1 < m && uniform(be > kPairNorm * hn);
            }
            double *wo = w1;
            if (pair) {
                // steps j and j + 1 share one Gram-Schmidt pass (as in
                // trl_run): w = s H w1 - al2 s w1 - be v_j with s = 1/be
                const double s = 1.0 / be;
                al2 = wg_hxv(t, w1, w);
                ++used;
                al2 = s * s * wg_sum(al2, sh);
                for (int e = threadIdx.x; e < n; e += kQBlock)
                    w[e] = s * w[e] - al2 * s * w1[e] - be * vj[e];
                __syncthreads();
                wg_dots<2>(t.Y, nl, V, j + 1, w1, w, n, sh.c, sh);
                nn = wg_subtract<2>(t.Y, nl, V, j + 1, w1, w, n, sh.c, s, sh);
                hn = fmax(hn, fmax(fabs(al2), sqrt(nn)));
                ++j;
                wo = w;
            }
            // a step by itself, and a remainder too small for the shared pass;
            // the coefficients on V[0..j] land in sh.A's first column as scratch
            double *cj = sh.A;
            if (!pair || !uniform(sqrt(nn) > kPairNorm * hn))
                nn = wg_orth(t.Y, nl, V, j + 1, wo, n, cj, sh);
            wg_normalize(V + (size_t)(j + 1) * n, wo, n, nn);
            const double bn = sqrt(nn);
            if (threadIdx.x == 0 && j >= 0) {
                if (pair) {
                    sh.T[(j - 1) * m + j - 1] = al;
                    sh.T[(j - 2) * m + j - 1] = sh.T[(j - 1) * m + j - 2] = beta_last;
                    sh.T[(j - 1) * m + j] = sh.T[j * m + j - 1] = be;
                    sh.T[j * m + j] = al2;
                } else {
                    if (j > k) {
                        cj[j] += al;
                        cj[j - 1] += beta_last;
                    }
                    for (int q = 0; q <= j; ++q) {
                        const bool arrow = (j == k) && (q < k);
                        if (arrow || q >= j - 1) sh.T[q * m + j] = sh.T[j * m + q] = cj[q];
                    }
                }
                if (j + 1 < m) sh.T[(j + 1) * m + j] = sh.T[j * m + j + 1] = bn;
            }
            if (j >= 0) {
                beta_last = bn;
                if (j > k) hn = fmax(hn, bn);
            }
            ++j;
            __syncthreads();
        }
        fresh = false;
        for (int e = threadIdx.x; e < m * m; e += kQBlock) sh.A[e] = sh.T[e];
        __syncthreads();
        wg_jacobi(m, sh);
        bool ok = true;
        for (int q = 0; q < want; ++q) {
            const double rn = full ? 0.0 : fabs(beta_last * sh.S[q * m + (m - 1)]);
            if (rn > 0.1 * tol * fmax(1.0, fabs(sh.theta[q]))) ok = false;
        }
        ok = uniform(ok);
        const bool last = ok || used >= maxit || full;
        // thick restart: kk Ritz vectors and the residual direction
        const int kk = last ? want : min(m - 2, want + max(1, (m - want) / 2));
        wg_rotate(V, Vs, n, m, kk, sh);
        double *x = V;
        V = Vs;
        Vs = x;
        if (last) {
            converged = ok || full;
            break;
        }
        wg_copy(V + (size_t)kk * n, Vs + (size_t)m * n, n);
        for (int e = threadIdx.x; e < m * m; e += kQBlock) sh.T[e] = 0.0;
        __syncthreads();
        if (threadIdx.x == 0)
            for (int q = 0; q < kk; ++q) {
                sh.T[q * m + q] = sh.theta[q];
                const double arrow = beta_last * sh.S[q * m + (m - 1)];
                sh.T[q * m + kk] = sh.T[kk * m + q] = arrow;
            }
        __syncthreads();
        k = kk;
    }
    for (int q = 0; q < want; ++q) {
        const double *vq = V + (size_t)q * n;
        wg_hxv(t, vq, w);
        const double th = sh.theta[q];
        double s = 0.0;
        for (int e = threadIdx.x; e < n; e += kQBlock) {
            const double r = w[e] - th * vq[e];
            s += r * r;
        }
        const double r = sqrt(wg_sum(s, sh));
        if (threadIdx.x == 0) {
            sh.th[q] = th;
            sh.rr[q] = r;
        }
        if (r > tol * fmax(1.0, fabs(th))) converged = false;
        wg_copy(t.X + (size_t)q * n, vq, n);
    }
    __syncthreads();
    return converged ? 0 : DMED_ENOCONV;
}

// The deflation rounds of trl_deflated, then the kept vectors in ascending
// energy to the task's outputs.
__device__ __forceinline__ void wg_solve(const SqTask &t, Shared &sh)
{
    const int n = t.dim, neig = t.neig;
    const int want = t.lowest ? 1 : neig;
    double *V = t.V, *Vs = t.Vs;
    int used = 0, rcfinal = 0, nk = 0;
    constexpr double confirm_tol = 1e-6;
    for (int round = 0; round <= neig; ++round) {
        const int nl = nk;
        if (n - nl < want) break;
        const uint64_t seed = 1234567ull + 7919ull * (uint64_t)round;
        // rounds after the first start with a loose solve, which settles most
        int rc = 0;
        bool reach = true;
        for (int tight = nl > 0 && confirm_tol > t.tol ? 0 : 1; tight < 2 && reach; ++tight) {
            rc = wg_trl(t, want, t.m, max(t.maxit - used, 4 * t.m), tight ? t.tol : confirm_tol, nl,
                        seed, V, Vs, used, sh);
            if (tight) break;
            reach = false;
            for (int q = 0; q < want; ++q) {
                const double lo = sh.th[q] - sh.rr[q];
                if (t.lowest ? (lo <= sh.ke[0] + t.degen) : (nk < neig || lo < sh.ke[nk - 1]))
                    reach = true;
            }
            reach = uniform(reach);
        }
        if (!reach) break;
        if (rc == DMED_ENOCONV) rcfinal = rc;
        bool added = false;
        for (int q = 0; q < want; ++q) {
            int slot = -1;
            if (threadIdx.x == 0) {
                const double e = sh.th[q], r = sh.rr[q];
                if (t.lowest) {
                    if (!(nk > 0 && !(e <= sh.ke[0] + t.degen)) && nk < neig) slot = nk;
                } else if (nk >= neig) {
                    // nothing new below the top, else evict the highest level
                    if (e < sh.ke[nk - 1]) {
                        slot = sh.kslot[nk - 1];
                        --nk;
                    }
                } else {
                    unsigned busy = 0u;
                    for (int i = 0; i < nk; ++i) busy |= 1u << sh.kslot[i];
                    slot = __ffs(~busy) - 1;
                }
                if (slot >= 0) {
                    // insert in ascending energy (stable after equal energies)
                    int i = nk;
                    while (i > 0 && sh.ke[i - 1] > e) {
                        sh.ke[i] = sh.ke[i - 1];
                        sh.kr[i] = sh.kr[i - 1];
                        sh.kslot[i] = sh.kslot[i - 1];
                        --i;
                    }
                    sh.ke[i] = e;
                    sh.kr[i] = r;
                    sh.kslot[i] = slot;
                    ++nk;
                }
                sh.ibcast = slot;
                sh.bcast = (double)nk;
            }
            __syncthreads();
            slot = __builtin_amdgcn_readfirstlane(sh.ibcast);
            nk = __builtin_amdgcn_readfirstlane((int)sh.bcast);
            __syncthreads();
            if (slot >= 0) {
                wg_copy(t.Y + (size_t)slot * n, t.X + (size_t)q * n, n);
                added = true;
            }
        }
        if (!added || used >= t.maxit) break;
        if (t.lowest && nk >= neig) break;
    }
    for (int q = 0; q < nk; ++q) wg_copy(t.evecs[q], t.Y + (size_t)sh.kslot[q] * n, n);
    if (threadIdx.x == 0) {
        for (int q = 0; q < nk; ++q) {
            t.evals[q] = sh.ke[q];
            t.resid[q] = sh.kr[q];
        }
        t.info[0] = nk;
        t.info[1] = rcfinal;
        t.info[2] = used;
    }
    __syncthreads();
}

__global__ void __launch_bounds__(kQBlock) k_sector_queue(const SqTask *__restrict__ tasks,
                                                          int ntask, int *__restrict__ counter)
{
    extern __shared__ __align__(16) unsigned char smem[];
    Shared &sh = *reinterpret_cast<Shared *>(smem);
    for (;;) {
        if (threadIdx.x == 0) sh.ibcast = atomicAdd(counter, 1);
        __syncthreads();
        const int k = __builtin_amdgcn_readfirstlane(sh.ibcast);
        __syncthreads();
        if (k >= ntask) break;
        const SqTask &t = tasks[k];
        wg_solve(t, sh);
    }
}

}  // namespace

// ------------------------------------------------------------------ host
int64_t queue_max_dim()
{
    static const int64_t d = [] {
        const char *e = std::getenv("DMED_SECTOR_QUEUE_MAXDIM");
        return e ? (int64_t)std::atoll(e) : kQueueMaxDim;
    }();
    return d;
}

bool queue_takes(const dmed_sector *s, int neig, int ncv)
{
    return s->jterms == 0 && s->dim <= queue_max_dim() && s->dim < (int64_t)1 << 30 &&
           neig >= 1 && neig <= kQMaxNeig &&
           neig < s->dim && std::max(ncv, neig + 2) <= kQMaxM + 8;
}

int queue_launch(SectorQueue &q, hipStream_t st)
{
    const int nt = (int)q.items.size();
    if (nt == 0) return 0;
    size_t words = 0;
    for (auto &it : q.items) {
        const int64_t n = it.s->dim;
        const int m = std::min(std::max(it.ncv, it.neig + 2), kQMaxM);
        words += (size_t)(2 * (m + 1) + 1 + 2 * it.neig) * n + 64;
    }
    DMED_HIP(hipMalloc(&q.work, words * 8));
    DMED_HIP(hipMalloc(&q.res, (size_t)nt * (2 * kQMaxNeig + 4) * 8));
    DMED_HIP(hipMalloc(&q.ptrs, (size_t)nt * kQMaxNeig * sizeof(double *)));
    DMED_HIP(hipMalloc(&q.counter, sizeof(int)));
    std::vector<SqTask> tasks(nt);
    std::vector<double *> ptrs((size_t)nt * kQMaxNeig, nullptr);
    double *wp = q.work;
    for (int k = 0; k < nt; ++k) {
        auto &it = q.items[k];
        const dmed_sector *s = it.s;
        const int64_t n = s->dim;
        const int m = std::min(std::max(it.ncv, it.neig + 2), kQMaxM);
        SqTask &t = tasks[k];
        t.hu_idx = s->up->hidx;
        t.hd_idx = s->dw->hidx;
        t.hu_val = s->up->hval;
        t.hd_val = s->dw->hval;
        t.du = s->up->diag;
        t.dd = s->dw->diag;
        t.W = s->W;
        t.impu = s->up->imp;
        t.impd = s->dw->imp;
        t.dup = (int32_t)s->up->dim;
        t.ddw = (int32_t)s->dw->dim;
        t.nhu = s->up->nhop;
        t.nhd = s->dw->nhop;
        t.nimp = s->nimp;
        t.dim = (int32_t)n;
        t.neig = it.neig;
        t.m = m;
        t.maxit = it.maxit;
        t.lowest = it.lowest ? 1 : 0;
        t.tol = it.tol;
        t.degen = it.degen;
        t.V = wp;
        wp += (size_t)(m + 1) * n;
        t.Vs = wp;
        wp += (size_t)(m + 1) * n;
        t.w = wp;
        wp += n;
        t.Y = wp;
        wp += (size_t)it.neig * n;
        t.X = wp;
        wp += (size_t)it.neig * n + 64;
        it.vecs.assign(it.neig, nullptr);
        for (int q = 0; q < it.neig; ++q) {
            dmed_vec *v = new dmed_vec{s, DMED_FP64, n, nullptr};
            if (hipMalloc(&v->data, (size_t)std::max<int64_t>(n, 1) * 8) != hipSuccess) {
                delete v;
                return fail(DMED_ENOMEM, "sector queue: eigenvector allocation");
            }
            it.vecs[q] = v;
            ptrs[(size_t)k * kQMaxNeig + q] = (double *)v->data;
        }
        t.evecs = q.ptrs + (size_t)k * kQMaxNeig;
        double *r = q.res + (size_t)k * (2 * kQMaxNeig + 4);
        t.evals = r;
        t.resid = r + kQMaxNeig;
        t.info = reinterpret_cast<int32_t *>(r + 2 * kQMaxNeig);
    }
    DMED_HIP(hipMalloc(&q.tasks, (size_t)nt * sizeof(SqTask)));
    DMED_HIP(hipMemcpyAsync(q.tasks, tasks.data(), (size_t)nt * sizeof(SqTask), hipMemcpyHostToDevice, st));
    DMED_HIP(hipMemcpyAsync(q.ptrs, ptrs.data(), ptrs.size() * sizeof(double *), hipMemcpyHostToDevice, st));
    DMED_HIP(hipMemsetAsync(q.counter, 0, sizeof(int), st));
    DMED_HIP(hipMemsetAsync(q.res, 0, (size_t)nt * (2 * kQMaxNeig + 4) * 8, st));
    DMED_HIP(hipStreamSynchronize(st));     // the host task tables go out of scope
    static_assert(sizeof(Shared) <= 160 * 1024, "queue LDS");
    if (int rc = [&]() -> int {
            static const hipError_t e = hipFuncSetAttribute(
                (const void *)k_sector_queue, hipFuncAttributeMaxDynamicSharedMemorySize,
                (int)sizeof(Shared));
            return e == hipSuccess ? 0 : fail(DMED_EHIP, "sector queue: LDS attribute");
        }())
        return rc;
    const int ncu = std::max(8, ctx().num_cu);
    const unsigned grid = (unsigned)std::min(nt, ncu);
    DMED_HIP(hipEventCreate(&q.ev0));
    DMED_HIP(hipEventCreate(&q.ev1));
    DMED_HIP(hipEventRecord(q.ev0, st));
    hipLaunchKernelGGL(k_sector_queue, dim3(grid), dim3(kQBlock), sizeof(Shared), st,
                       (const SqTask *)q.tasks, nt, q.counter);
    DMED_HIP(hipGetLastError());
    DMED_HIP(hipEventRecord(q.ev1, st));
    q.stream = st;
    return 0;
}

int queue_finish(SectorQueue &q)
{
    const int nt = (int)q.items.size();
    int rc = 0;
    if (nt > 0 && q.stream) {
        std::vector<double> res((size_t)nt * (2 * kQMaxNeig + 4));
        if (hipMemcpyAsync(res.data(), q.res, res.size() * 8, hipMemcpyDeviceToHost, q.stream) !=
                hipSuccess ||
            hipStreamSynchronize(q.stream) != hipSuccess)
            rc = fail(DMED_EHIP, "sector queue: result copy");
        if (!rc && hipEventElapsedTime(&q.kernel_ms, q.ev0, q.ev1) != hipSuccess) q.kernel_ms = -1.f;
        for (int k = 0; k < nt && !rc; ++k) {
            auto &it = q.items[k];
            const double *r = res.data() + (size_t)k * (2 * kQMaxNeig + 4);
            int32_t info[3];
            std::memcpy(info, r + 2 * kQMaxNeig, sizeof info);
            it.nout = info[0];
            it.rc = info[1];
            it.used = info[2];
            it.evals.assign(r, r + it.nout);
            it.resid.assign(r + kQMaxNeig, r + kQMaxNeig + it.nout);
            for (int q2 = it.nout; q2 < it.neig; ++q2) {
                dmed_vec_free(it.vecs[q2]);
                it.vecs[q2] = nullptr;
            }
            it.vecs.resize(it.nout);
        }
    }
    if (nt > 0 && !q.stream)        // never launched: drop the eigenvector buffers
        for (auto &it : q.items) {
            for (dmed_vec *v : it.vecs) dmed_vec_free(v);
            it.vecs.clear();
            it.nout = 0;
            it.rc = DMED_EHIP;
        }
    if (q.ev0) hipEventDestroy(q.ev0);
    if (q.ev1) hipEventDestroy(q.ev1);
    q.ev0 = q.ev1 = nullptr;
    hipFree(q.work);
    hipFree(q.res);
    hipFree(q.ptrs);
    hipFree(q.counter);
    hipFree(q.tasks);
    q.work = q.res = nullptr;
    q.ptrs = nullptr;
    q.counter = nullptr;
    q.tasks = nullptr;
    q.stream = nullptr;
    return rc;
}

}  // namespace dmed
