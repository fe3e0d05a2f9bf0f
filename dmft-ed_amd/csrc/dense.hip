// dense.hip -- dense eigen-decompositions of small sectors on the device.
//
// Sectors up to lanc_dim_threshold states are diagonalised in full
// (ED_DIAG.f90:185-193).  On the host each costs O(n^3) on one thread (16 to
// 24 ms at 225 states), and a small bath is mostly such sectors.  Here one
// launch takes all of a solve's: one workgroup per sector builds H from the
// sector tables, reduces it to tridiagonal form by Householder reflections,
// runs the implicit QL iteration, and transforms the wanted eigenvectors back
// -- the algorithm of host_syev (hostla.cpp).
//
// Measured on a T = 0 solve at Ns = 6 (21 dense sectors of up to 225 states
// beside four Krylov sectors): 101 -> 30 ms.
//
// Bounds: the reduction streams the trailing matrix from L2 three times a
// step (2.9 ms of the 12 ms at 225 states, eight columns in flight); the QL
// recurrence is serial, so wave 0 runs it one sweep ahead of the other waves,
// which apply the rotations of the sweep before to the rows of Z (a lane per
// row, coalesced along the column).  Z and H stay in the
// XCD's L2 (2 x 405 KB at 225 states).
#include <algorithm>
#include <cmath>
#include <vector>

#include "dmed_internal.h"
#include "tridiag_device.h"

namespace dmed {

int lds_attr_once(const void *kern);

namespace {

constexpr int kDenseBlock = 1024;
constexpr int kDenseWaves = kDenseBlock / 64;

struct DenseTask {
    const int32_t *hu_idx, *hd_idx, *ju, *jd;
    const double *hu_val, *hd_val, *du, *dd, *W;
    const uint8_t *impu, *impd;
    int32_t dup, ddw, nhu, nhd, nimp, jterms, norb, n, neig;
    double jx, jp;
    double *A, *Z;                      // n*n each
    double *vecs, *evals;               // neig*n, neig
    int32_t *status;
};

__device__ __forceinline__ double wsum_all(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// workgroup sum, the same value in every lane; red: kDenseWaves doubles
__device__ __forceinline__ double dsum(double v, double *red)
{
    v = wsum_all(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kDenseWaves; ++w) s += red[w];
    return s;
}

// Place of level i among d[0..n): ascending, equal levels by index, and levels
// that are not a number after all others, by index.  A total order, so that
// the places of all levels are 0..n-1 each once, whatever d holds.
__host__ __device__ inline int level_place(const double *d, int n, int i)
{
    const double x = d[i];
    int p = 0;
    for (int j = 0; j < n; ++j) {
        const double y = d[j];
        const bool before = x == x ? y < x || (y == x && j < i) : y == y || j < i;
        p += before ? 1 : 0;
    }
    return p;
}

// H of the sector into A (column-major), a row per lane: the terms of
// k_hxv's row sum
__device__ void build_h(const DenseTask &t)
{
    const int n = t.n, dup = t.dup, ddw = t.ddw;
    double *A = t.A;
    for (int e = threadIdx.x; e < n * n; e += kDenseBlock) A[e] = 0.0;
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += kDenseBlock) {
        const int id = i / dup, iu = i - id * dup;
        A[i * n + i] += t.du[iu] + t.dd[id] + t.W[t.impu[iu] * t.nimp + t.impd[id]];
        for (int h = 0; h < t.nhu; ++h)
            A[(t.hu_idx[h * dup + iu] + id * dup) * n + i] += t.hu_val[h * dup + iu];
        for (int h = 0; h < t.nhd; ++h)
            A[(iu + t.hd_idx[h * ddw + id] * dup) * n + i] += t.hd_val[h * ddw + id];
        if (!t.jterms) continue;
        const int no = t.norb;
        for (int pa = 0; pa < no; ++pa)
            for (int pb = 0; pb < no; ++pb) {
                if (pa == pb) continue;
                const int wu = t.ju[(pa * no + pb) * dup + iu];
                if (wu < 0) continue;
                const double su = (wu & 1) ? -1.0 : 1.0;
                const int wx = t.jd[(pb * no + pa) * ddw + id];
                if (wx >= 0)
                    A[((wu >> 1) + (wx >> 1) * dup) * n + i] += t.jx * su * ((wx & 1) ? -1.0 : 1.0);
                const int wp = t.jd[(pa * no + pb) * ddw + id];
                if (wp >= 0)
                    A[((wu >> 1) + (wp >> 1) * dup) * n + i] += t.jp * su * ((wp & 1) ? -1.0 : 1.0);
            }
    }
    __syncthreads();
}

// LDS: eight arrays of n doubles and the reduction buffers
__global__ void __launch_bounds__(kDenseBlock) k_dense_eigh(const DenseTask *__restrict__ tasks)
{
    extern __shared__ double sm[];
    __shared__ double red[kDenseWaves];
    __shared__ double part[kDenseBlock];
    __shared__ double sink[kQlSink];
    __shared__ double scale;
    __shared__ int pub[2][3];           // per rotation buffer: l, m, more
    __shared__ int bad;
    const DenseTask t = tasks[blockIdx.x];
    const int n = t.n, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    double *d = sm, *e = d + n, *v = e + n, *q = v + n, *rc0 = q + n, *rs0 = rc0 + n, *rc1 = rs0 + n,
           *rs1 = rc1 + n;
    double *A = t.A, *Z = t.Z;
    build_h(t);
    for (int i = tid; i < n; i += kDenseBlock) e[i] = 0.0;
    if (tid == 0) bad = 0;
    // column groups of the reduction's passes: lane -> row and group
    const int gl = n >= kDenseBlock ? kDenseBlock : n;          // lanes a group
    const int ng = kDenseBlock / gl, grp = tid / gl, row0 = tid - grp * gl;
    __syncthreads();
    // Householder reduction: reflector k (v, scaled by sqrt(c)) stays in
    // column k below the diagonal
    for (int k = 0; k + 2 < n; ++k) {
        double *ck = A + (size_t)k * n;
        double s = 0.0;
        for (int i = k + 2 + tid; i < n; i += kDenseBlock) s += ck[i] * ck[i];
        const double tail = dsum(s, red);
        const double x0 = ck[k + 1];
        if (tid == 0) d[k] = ck[k];
        if (tail == 0.0) {                                      // column already reduced
            if (tid == 0) e[k] = x0;
            __syncthreads();
            for (int i = k + 1 + tid; i < n; i += kDenseBlock) ck[i] = 0.0;
            __syncthreads();
            continue;
        }
        const double nrm = sqrt(tail + x0 * x0), alpha = x0 > 0.0 ? -nrm : nrm;
        const double v0 = x0 - alpha, sc = sqrt(2.0 / (tail + v0 * v0));
        if (tid == 0) e[k] = alpha;
        __syncthreads();
        for (int i = k + 1 + tid; i < n; i += kDenseBlock) {
            const double x = sc * (i == k + 1 ? v0 : ck[i]);
            v[i] = x;
            ck[i] = x;
        }
        __syncthreads();
        // q = B v over the trailing block, then q -= (v.q/2) v
        for (int i0 = 0; i0 < n; i0 += gl) {
            const int i = i0 + row0;
            double acc = 0.0;
            // eight columns in flight (unconditional loads at clamped indices)
            if (grp < ng && i < n && i > k)
                for (int j0 = k + 1 + grp; j0 < n; j0 += 8 * ng) {
                    double a[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) a[u] = A[min(j0 + u * ng, n - 1) * n + i];
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        if (j0 + u * ng < n) acc += a[u] * v[j0 + u * ng];
                }
            if (ng > 1) {
                part[tid] = acc;
                __syncthreads();
                if (grp == 0 && i < n) {
                    for (int g = 1; g < ng; ++g) acc += part[g * gl + row0];
                    q[i] = acc;
                }
                __syncthreads();
            } else if (grp == 0 && i < n) {
                q[i] = acc;
            }
        }
        __syncthreads();
        s = 0.0;
        for (int i = k + 1 + tid; i < n; i += kDenseBlock) s += v[i] * q[i];
        const double half = 0.5 * dsum(s, red);
        for (int i = k + 1 + tid; i < n; i += kDenseBlock) q[i] -= half * v[i];
        __syncthreads();
        for (int i0 = 0; i0 < n; i0 += gl) {
            const int i = i0 + row0;
            if (grp < ng && i < n && i > k) {
                const double vi = v[i], qi = q[i];
                for (int j0 = k + 1 + grp; j0 < n; j0 += 8 * ng) {
                    double a[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) a[u] = A[min(j0 + u * ng, n - 1) * n + i];
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        const int j = j0 + u * ng;
                        if (j < n) A[j * n + i] = a[u] - (vi * q[j] + qi * v[j]);
                    }
                }
            }
        }
        __syncthreads();
    }
    if (tid == 0) {
        if (n > 1) {
            d[n - 2] = A[(size_t)(n - 2) * n + n - 2];
            e[n - 2] = A[(size_t)(n - 2) * n + n - 1];
        }
        d[n - 1] = A[(size_t)(n - 1) * n + n - 1];
        e[n - 1] = 0.0;
    }
    for (int x = tid; x < n * n; x += kDenseBlock) Z[x] = (x % n == x / n) ? 1.0 : 0.0;
    __syncthreads();
    if (wave == 0) {
        const double sc = ql_scale(d, e, n);
        if (lane == 0) scale = sc;
        for (int i = lane; i < n; i += 64) {
            d[i] *= sc;
            e[i] *= sc;
        }
    }
    __syncthreads();
    // QL: in turn `it`, wave 0 computes sweep it into buffer it&1 while the
    // others apply sweep it - 1 from the other buffer
    int l = 0, m = 0, iter = 0;
    bool inside = false;
    double f = 0.0, tst1 = 0.0;
    for (int it = 0;; ++it) {
        double *rc = (it & 1) ? rc1 : rc0, *rs = (it & 1) ? rs1 : rs0;
        if (wave == 0) {
            int more = 0;
            while (l < n) {
                if (!inside) {
                    tst1 = fmax(tst1, fabs(d[l]) + fabs(e[l]));
                    m = ql_find(e, n, l, tst1);
                    iter = 0;
                    inside = m != l;
                }
                if (inside && iter >= 30) {
                    if (lane == 0) bad = 1;
                    l = n;
                    break;
                }
                if (inside) {
                    const double el = ql_iterate<true>(d, e, n, l, m, f, rc, rs, nullptr, sink);
                    ++iter;
                    more = 1;
                    if (lane == 0) {
                        pub[it & 1][0] = l;
                        pub[it & 1][1] = m;
                    }
                    if (tst1 + el > tst1) break;                // not converged: one sweep a turn
                    inside = false;
                }
                wave_lds_fence();
                if (lane == 0) d[l] += f;
                wave_lds_fence();
                ++l;
                if (more) break;
            }
            if (lane == 0) pub[it & 1][2] = more;
        } else if (it > 0) {
            const int pl = pub[(it - 1) & 1][0], pm = pub[(it - 1) & 1][1];
            const double *pc = (it & 1) ? rc0 : rc1, *ps = (it & 1) ? rs0 : rs1;
            for (int r = tid - 64; r < n; r += kDenseBlock - 64) {
                double *zr = Z + r;
                double zn = zr[(size_t)pm * n];
                int i = pm - 1;
                // eight columns loaded ahead of their rotations
                for (; i - 7 >= pl; i -= 8) {
                    double z[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) z[u] = zr[(size_t)(i - u) * n];
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        const double c = pc[i - u], s = ps[i - u];
                        zr[(size_t)(i - u + 1) * n] = s * z[u] + c * zn;
                        zn = c * z[u] - s * zn;
                    }
                }
                for (; i >= pl; --i) {
                    const double c = pc[i], s = ps[i], zi = zr[(size_t)i * n];
                    zr[(size_t)(i + 1) * n] = s * zi + c * zn;
                    zn = c * zi - s * zn;
                }
                zr[(size_t)pl * n] = zn;
            }
        }
        __syncthreads();
        if (!pub[it & 1][2]) break;
    }
    // ascending selection of the wanted eigenvalues; a level that is not finite
    // (a model with NaN or infinity) is reported like one that did not converge
    int *order = reinterpret_cast<int *>(v);
    for (int i = tid; i < n; i += kDenseBlock) {
        order[level_place(d, n, i)] = i;
        if (!isfinite(d[i])) bad = 1;
    }
    __syncthreads();
    // back-transformation, a wave per eigenvector: y -= v_k (v_k . y)
    for (int w = wave; w < t.neig; w += kDenseWaves) {
        const double *z = Z + (size_t)order[w] * n;
        double *y = t.vecs + (size_t)w * n;
        for (int i = lane; i < n; i += 64) y[i] = z[i];
        for (int k = n - 3; k >= 0; --k) {
            const double *vk = A + (size_t)k * n;
            double s = 0.0;
            for (int i = lane; i < n; i += 64) s += i > k ? vk[i] * y[i] : 0.0;
            s = wsum_all(s);
            for (int i = lane; i < n; i += 64)
                if (i > k) y[i] -= s * vk[i];
        }
        if (lane == 0) t.evals[w] = d[order[w]] / scale;
    }
    if (tid == 0) *t.status = bad;
}

}  // namespace

bool dense_takes(int64_t n) { return n >= 1 && n <= kDenseMaxDim; }

// order[q] = index of the q-th level, by the rule of k_dense_eigh
void dense_order(int n, const double *d, int *order)
{
    for (int i = 0; i < n; ++i) order[level_place(d, n, i)] = i;
}

// Launch the items on e's stream (asynchronous); dense_finish waits.
// DMED_ENOMEM: no room for the work space, nothing was launched.
int dense_launch(DenseBatch &b, Exec &e)
{
    b.exec = &e;
    const size_t nt = b.items.size();
    if (nt == 0) return 0;
    auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
    size_t off = up(nt * sizeof(DenseTask));
    const size_t ores = off;                    // eigenvalues and states: one download
    size_t nev = 0;
    int64_t nmax = 1;
    for (const DenseItem &it : b.items) {
        nev += it.neig;
        nmax = std::max(nmax, it.s->dim);
    }
    off += up(nev * 8 + nt * 4);
    std::vector<size_t> at(nt);
    for (size_t k = 0; k < nt; ++k) {
        const size_t n = (size_t)b.items[k].s->dim;
        at[k] = off;
        off += up(2 * n * n * 8) + up((size_t)b.items[k].neig * n * 8);
    }
    unsigned char *d = nullptr;
    if (int rc = exec_try(e, kSlotDense, off, (void **)&d)) return rc;
    b.tasks.resize(nt * sizeof(DenseTask));
    DenseTask *h = reinterpret_cast<DenseTask *>(b.tasks.data());
    double *dev = reinterpret_cast<double *>(d + ores);
    int32_t *dst = reinterpret_cast<int32_t *>(dev + nev);
    size_t e0 = 0;
    for (size_t k = 0; k < nt; ++k) {
        DenseItem &it = b.items[k];
        const dmed_sector *s = it.s;
        DenseTask &t = h[k];
        t.hu_idx = s->up->hidx;
        t.hd_idx = s->dw->hidx;
        t.hu_val = s->up->hval;
        t.hd_val = s->dw->hval;
        t.ju = s->up->ipair;
        t.jd = s->dw->ipair;
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
        t.jterms = s->jterms;
        t.norb = s->norb;
        t.n = (int32_t)s->dim;
        t.neig = it.neig;
        t.jx = s->jx;
        t.jp = s->jp;
        const size_t n = (size_t)s->dim;
        t.A = reinterpret_cast<double *>(d + at[k]);
        t.Z = t.A + n * n;
        t.vecs = reinterpret_cast<double *>(d + at[k] + up(2 * n * n * 8));
        t.evals = dev + e0;
        t.status = dst + k;
        it.dvecs = t.vecs;
        e0 += it.neig;
    }
    DMED_HIP(hipMemcpyAsync(d, h, nt * sizeof(DenseTask), hipMemcpyHostToDevice, e.stream));
    const size_t lds = 8 * (size_t)nmax * 8;
    if (int rc = lds_attr_once((const void *)k_dense_eigh)) return rc;
    hipLaunchKernelGGL(k_dense_eigh, dim3((unsigned)nt), dim3(kDenseBlock), lds, e.stream,
                       reinterpret_cast<const DenseTask *>(d));
    DMED_HIP(hipGetLastError());
    b.dres = dev;
    b.nev = nev;
    return 0;
}

int dense_finish(DenseBatch &b)
{
    const size_t nt = b.items.size();
    if (nt == 0 || !b.dres) return 0;
    hipStream_t st = b.exec->stream;
    std::vector<double> res(b.nev + (nt * 4 + 7) / 8);
    DMED_HIP(hipMemcpyAsync(res.data(), b.dres, b.nev * 8 + nt * 4, hipMemcpyDeviceToHost, st));
    DMED_HIP(hipStreamSynchronize(st));
    const int32_t *status = reinterpret_cast<const int32_t *>(res.data() + b.nev);
    size_t e0 = 0;
    for (size_t k = 0; k < nt; ++k) {
        DenseItem &it = b.items[k];
        it.evals.assign(res.begin() + e0, res.begin() + e0 + it.neig);
        e0 += it.neig;
        it.rc = status[k] ? DMED_ENOCONV : 0;
        it.nout = it.neig;
        // the lowest level and its copies, where nothing else is wanted
        if (it.lowest)
            for (it.nout = 1; it.nout < it.neig && it.evals[it.nout] <= it.evals[0] + it.degen;)
                ++it.nout;
        if (it.rc || !it.want_vecs) continue;
        const size_t n = (size_t)it.s->dim;
        for (int q = 0; q < it.nout; ++q) {
            dmed_vec *v = new dmed_vec{it.s, DMED_FP64, it.s->dim, nullptr};
            it.vecs.push_back(v);
            DMED_HIP(hipMalloc(&v->data, n * 8));
            DMED_HIP(hipMemcpyAsync(v->data, it.dvecs + (size_t)q * n, n * 8, hipMemcpyDeviceToDevice, st));
        }
    }
    DMED_HIP(hipStreamSynchronize(st));
    return 0;
}

}  // namespace dmed
