// chainwg.hip -- Lanczos chain of a small sector in one workgroup.
//
// A chain step of a few thousand states is far too small for the chip: as
// four launches (H*v, alpha, update, beta) it costs about 8 us however few
// states there are, and a solve runs hundreds of such chains.  Here one
// workgroup runs all the steps of a chain in one launch.  The Lanczos vector
// lives in LDS, the previous one in registers, and the scalars in every
// lane, so a step costs two barriers and no memory traffic beyond LDS.
//
// Lane layout: a lane keeps one row iu of the D_up x D_dw matrix and the
// columns g, g + G, g + 2G, .. (G = lanes / D_up column groups), at most R of
// them.  Its up hops (target row and coefficient) and the diagonal of its
// elements then serve all its columns, the down hops of a column are the same
// for all its lanes (LDS broadcasts), and both gathers read LDS with lanes
// along consecutive rows.  Bound by the LDS gathers.  Measured per FP64 step,
// as four launches -> here: 12.7 -> 1.3 us (100 states), 15.1 -> 2.5 us
// (1,225), 15.4 -> 3.9 us (4,900), 17.4 -> 6.7 us (7,056).
//
// The recurrence and its scalars are those of the launches in krylov.hip
// (k_hxv in Lanczos mode, k_chain_alpha, k_chain_update, k_chain_beta, k_accum);
// only the order of the reductions differs.
#include <algorithm>
#include <vector>

#include "dmed_internal.h"
#include "wave_device.h"

namespace dmed {

int lds_attr_once(const void *kern);

namespace {

template <typename T>
struct WgArgs {
    T *vp, *v;                          // previous and current vector, in and out
    int32_t dup, ddw, nhu, nhd, nimp, groups, count;
    const int32_t *hu_idx, *hd_idx;
    const T *hu_val, *hd_val;
    const double *du, *dd, *W;
    const uint8_t *impu, *impd;
    const int32_t *ju, *jd;             // impurity pair hops (jterms)
    int32_t norb;
    double jx, jp;
    ChainScalars *cs;
    double *alpha, *beta;
    double *psi;                        // with psi: psi += z_k v_k, step by step
    const double *z;
    int32_t r, nlanc;                   // batch: columns per lane, chain length
    double thr;
};

// LDS: the wave sums of a step's two reductions, the vector, and the hop
// tables (values, then offsets).  JT: with spin exchange and pair hopping.
// FRESH: a whole chain from the vector at v, which stays as it is: the first
// scale, the cleared coefficients and the scalars are made here.
template <typename T, int R, bool JT, bool FRESH>
__device__ __forceinline__ void chain_wg(const WgArgs<T> &a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int dup = a.dup, ddw = a.ddw, n = dup * ddw, nhu = a.nhu, nhd = a.nhd, G = a.groups;
    const int nw = blockDim.x >> 6, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double *red = reinterpret_cast<double *>(smem);              // [3][16]
    T *x = reinterpret_cast<T *>(smem + 3 * 16 * sizeof(double));
    T *huv = x + n, *hdv = huv + nhu * dup;
    int32_t *huo = reinterpret_cast<int32_t *>(hdv + nhd * ddw), *hdo = huo + nhu * dup;
    ChainScalars cs{};
    if constexpr (!FRESH) {
        cs = *a.cs;
        if (cs.done) return;
    }
    double s = 0.0;
    for (int e = threadIdx.x; e < n; e += blockDim.x) {
        const T v = a.v[e];
        x[e] = v;
        if constexpr (FRESH) s += (double)v * (double)v;
    }
    if constexpr (FRESH) {
        for (int k = threadIdx.x; k < a.nlanc; k += blockDim.x) a.alpha[k] = a.beta[k] = 0.0;
        s = wave_sum63(s);
        if (lane == 63) red[32 + wave] = s;     // written again only two barriers on
    }
    for (int e = threadIdx.x; e < nhu * dup; e += blockDim.x) {
        huv[e] = a.hu_val[e];
        huo[e] = a.hu_idx[e];
    }
    for (int e = threadIdx.x; e < nhd * ddw; e += blockDim.x) {
        hdv[e] = a.hd_val[e];
        hdo[e] = a.hd_idx[e] * dup;
    }
    // the lane's row and columns; lanes past the last group and columns past
    // the last repeat a valid element and are masked out
    const int g = threadIdx.x / dup;
    const bool lane_on = g < G;
    const int iu = threadIdx.x - g * dup;
    const int g0 = lane_on ? g : 0;
    T diag[R], vp[R], y[R];
    int id[R];
    const double du = a.du[iu];
    const int bu = a.impu[iu] * a.nimp;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        id[r] = min(g0 + r * G, ddw - 1);
        const int c = id[r];
        diag[r] = (T)(du + (a.dd[c] + a.W[bu + a.impd[c]]));
        if constexpr (FRESH)
            vp[r] = 0;
        else
            vp[r] = a.vp[c * dup + iu];
    }
    __syncthreads();
    if constexpr (FRESH) {
        s = 0.0;
        for (int w = 0; w < nw; ++w) s += red[32 + w];
        cs.sx = 1.0 / sqrt(s);
        cs.thr = a.thr;
        cs.done = s == 0.0 ? 1 : 0;
        cs.nlanc = a.nlanc;
    }
    for (int it = 0; it < a.count && !cs.done; ++it) {
        if (!FRESH && a.psi) {
            const double c = a.z[cs.step] * cs.sx;
#pragma unroll 1
            for (int e = threadIdx.x; e < n; e += blockDim.x) a.psi[e] += c * (double)x[e];
        }
#pragma unroll
        for (int r = 0; r < R; ++r) y[r] = diag[r] * x[id[r] * dup + iu];
#pragma unroll 1
        for (int h = 0; h < nhu; ++h) {
            const int j = huo[h * dup + iu];
            const T v = huv[h * dup + iu];
#pragma unroll
            for (int r = 0; r < R; ++r) y[r] += v * x[id[r] * dup + j];
        }
#pragma unroll 1
        for (int h = 0; h < nhd; ++h) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int q = h * ddw + id[r];
                y[r] += hdv[q] * x[hdo[q] + iu];
            }
        }
        // spin exchange and pair hopping, as in k_hxv
        if constexpr (JT) {
            const int no = a.norb;
            for (int pa = 0; pa < no; ++pa)
                for (int pb = 0; pb < no; ++pb) {
                    if (pa == pb) continue;
                    const int wu = a.ju[(pa * no + pb) * dup + iu];
                    if (wu < 0) continue;
                    const int iu2 = wu >> 1;
                    const double su = (wu & 1) ? -1.0 : 1.0;
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const int wx = a.jd[(pb * no + pa) * ddw + id[r]];
                        if (wx >= 0)
                            y[r] += (T)(a.jx * su * ((wx & 1) ? -1.0 : 1.0)) * x[(wx >> 1) * dup + iu2];
                        const int wp = a.jd[(pa * no + pb) * ddw + id[r]];
                        if (wp >= 0)
                            y[r] += (T)(a.jp * su * ((wp & 1) ? -1.0 : 1.0)) * x[(wp >> 1) * dup + iu2];
                    }
                }
        }
        // alpha = sx*(<v, y> - b*svp*<v, v_prev>)
        double s0 = 0.0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            y[r] = (T)(cs.sx * (double)y[r]);
            if (lane_on && g + r * G < ddw) s0 += (double)x[id[r] * dup + iu] * (double)y[r];
        }
        s0 = wave_sum63(s0);
        if (lane == 63) red[wave] = s0;
        __syncthreads();                // no lane gathers from x past this point
        s0 = 0.0;
        for (int w = 0; w < nw; ++w) s0 += red[w];
        const double al = cs.sx * (s0 - cs.b * cs.svp * cs.q);
        const double ca = al * cs.sx, cb = cs.b * cs.svp;
        double s1 = 0.0, s2 = 0.0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const T xo = x[id[r] * dup + iu];
            const T w = (T)((double)y[r] - cb * (double)vp[r] - ca * (double)xo);
            vp[r] = xo;
            y[r] = w;
            if (lane_on && g + r * G < ddw) {
                s1 += (double)w * (double)w;
                s2 += (double)w * (double)xo;
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (lane_on && g + r * G < ddw) x[id[r] * dup + iu] = y[r];
        s1 = wave_sum63(s1);
        s2 = wave_sum63(s2);
        if (lane == 63) {
            red[16 + wave] = s1;
            red[32 + wave] = s2;
        }
        __syncthreads();
        s1 = 0.0;
        s2 = 0.0;
        for (int w = 0; w < nw; ++w) {
            s1 += red[16 + w];
            s2 += red[32 + w];
        }
        const double b = sqrt(s1);
        const int k = cs.step;
        if (threadIdx.x == 0) {
            a.alpha[k] = al;
            if (k + 1 < cs.nlanc) a.beta[k + 1] = b;
        }
        cs.alpha = al;
        cs.b = b;
        cs.q = s2;
        cs.svp = cs.sx;
        cs.sx = 1.0 / b;
        cs.step = k + 1;
        if (fabs(b) < cs.thr || k + 1 >= cs.nlanc) cs.done = 1;
    }
    if constexpr (!FRESH) {
        for (int e = threadIdx.x; e < n; e += blockDim.x) a.v[e] = x[e];
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (lane_on && g + r * G < ddw) a.vp[id[r] * dup + iu] = vp[r];
        if (threadIdx.x == 0) *a.cs = cs;
    }
}

template <typename T, int R, bool JT>
__global__ void __launch_bounds__(1024) k_chain_wg(const WgArgs<T> a)
{
    chain_wg<T, R, JT, false>(a);
}

// Many chains in one launch, one workgroup each: a solve has tens to hundreds
// of them, and launched one by one they share a few hardware queues and pay
// seven launches and copies each.  Green's functions and susceptibilities of
// an Ns = 8 solve with six states (about 110 chains): 50 -> 25 ms.
template <bool JT>
__global__ void __launch_bounds__(1024) k_chain_wg_batch(const WgArgs<double> *__restrict__ args)
{
    const WgArgs<double> &a = args[blockIdx.x];
    switch (a.r) {
    case 1: chain_wg<double, 1, JT, true>(a); break;
    case 2: chain_wg<double, 2, JT, true>(a); break;
    case 3: chain_wg<double, 3, JT, true>(a); break;
    case 4: chain_wg<double, 4, JT, true>(a); break;
    case 5: chain_wg<double, 5, JT, true>(a); break;
    case 6: chain_wg<double, 6, JT, true>(a); break;
    case 7: chain_wg<double, 7, JT, true>(a); break;
    case 8: chain_wg<double, 8, JT, true>(a); break;
    }
}

struct WgShape {
    int bs = 0, groups = 0, r = 0;
    size_t lds = 0;
};

// Launch shape of the one-workgroup chain, bs = 0 where it does not apply:
// a row per lane needs D_up <= 1024, and at most eight columns per lane keep
// the previous vector, the products and the diagonal in registers.  Small
// sectors take few lanes (cheaper barriers) as long as each has one or two
// columns.  At eight columns a step costs 8 us against the launches' 17;
// sectors past that would spill the registers.
WgShape wg_shape(const dmed_sector *s, int prec)
{
    WgShape w;
    const int64_t dup = s->up->dim, ddw = s->dw->dim;
    if (s->dim < 1 || s->dim > kChainWgMaxDim || dup > 1024) return w;
    const size_t esz = prec == DMED_FP32 ? 4 : 8;
    w.lds = 3 * 16 * 8 + (size_t)s->dim * esz + ((size_t)s->up->nhop * dup + (size_t)s->dw->nhop * ddw) * (esz + 4);
    if (w.lds + 1024 > ctx().lds_max) return w;
    for (int bs : {256, 512, 1024}) {
        if (dup > bs) continue;
        const int g = (int)std::min<int64_t>(bs / dup, ddw);
        const int r = (int)((ddw + g - 1) / g);
        if (r > 8 || (r > 2 && bs < 1024)) continue;
        w.bs = bs;
        w.groups = g;
        w.r = r;
        break;
    }
    return w;
}

template <typename T>
WgArgs<T> wg_args(const dmed_sector *s, const WgShape &w)
{
    WgArgs<T> a{};
    a.dup = (int32_t)s->up->dim;
    a.ddw = (int32_t)s->dw->dim;
    a.nhu = s->up->nhop;
    a.nhd = s->dw->nhop;
    a.nimp = s->nimp;
    a.groups = w.groups;
    a.r = w.r;
    a.hu_idx = s->up->hidx;
    a.hd_idx = s->dw->hidx;
    if constexpr (sizeof(T) == 8) {
        a.hu_val = s->up->hval;
        a.hd_val = s->dw->hval;
    } else {
        a.hu_val = s->up->hval32;
        a.hd_val = s->dw->hval32;
    }
    a.du = s->up->diag;
    a.dd = s->dw->diag;
    a.W = s->W;
    a.impu = s->up->imp;
    a.impd = s->dw->imp;
    a.ju = s->up->ipair;
    a.jd = s->dw->ipair;
    a.norb = s->norb;
    a.jx = s->jx;
    a.jp = s->jp;
    return a;
}

template <typename T, int R>
int launch_wg(const dmed_sector *s, const WgShape &w, void *vp, void *v, int count, ChainScalars *cs,
              double *alpha, double *beta, double *psi, const double *z, hipStream_t st)
{
    WgArgs<T> a = wg_args<T>(s, w);
    a.vp = static_cast<T *>(vp);
    a.v = static_cast<T *>(v);
    a.count = count;
    a.cs = cs;
    a.alpha = alpha;
    a.beta = beta;
    a.psi = psi;
    a.z = z;
    const auto kern = s->jterms ? k_chain_wg<T, R, true> : k_chain_wg<T, R, false>;
    if (int rc = lds_attr_once((const void *)kern)) return rc;
    hipLaunchKernelGGL(kern, dim3(1), dim3(w.bs), w.lds, st, a);
    DMED_HIP(hipGetLastError());
    return 0;
}

template <typename T>
int launch_wg_r(const dmed_sector *s, const WgShape &w, void *vp, void *v, int count,
                ChainScalars *cs, double *alpha, double *beta, double *psi, const double *z,
                hipStream_t st)
{
    switch (w.r) {
#define DMED_WG(R) \
    case R: return launch_wg<T, R>(s, w, vp, v, count, cs, alpha, beta, psi, z, st);
        DMED_WG(1) DMED_WG(2) DMED_WG(3) DMED_WG(4) DMED_WG(5) DMED_WG(6) DMED_WG(7) DMED_WG(8)
#undef DMED_WG
    }
    return fail(DMED_EINVAL, "one-workgroup chain: unsupported columns per lane");
}

}  // namespace

bool chain_wg_takes(const dmed_sector *s, int prec) { return wg_shape(s, prec).bs > 0; }

int chain_wg_steps(const dmed_sector *s, void *vp, void *v, int prec, int count, ChainScalars *cs,
                   double *alpha, double *beta, double *psi, const double *z, hipStream_t st)
{
    const WgShape w = wg_shape(s, prec);
    if (w.bs == 0) return fail(DMED_EINVAL, "sector too large for the one-workgroup chain");
    return prec == DMED_FP32 ? launch_wg_r<float>(s, w, vp, v, count, cs, alpha, beta, psi, z, st)
                             : launch_wg_r<double>(s, w, vp, v, count, cs, alpha, beta, psi, z, st);
}

bool chain_batch_takes(const dmed_sector *s, int nlanc)
{
    return nlanc > 0 && nlanc <= kChainMax && chain_wg_takes(s, DMED_FP64);
}

int chain_batch_run(std::vector<ChainBatchItem> &items, double threshold)
{
    if (items.empty()) return 0;
    // sectors with and without spin exchange take kernels of their own
    const auto jt = [](const ChainBatchItem &it) { return it.s->jterms != 0; };
    const auto mid = std::stable_partition(items.begin(), items.end(), jt);
    if (mid != items.begin() && mid != items.end()) {
        std::vector<ChainBatchItem> plain(mid, items.end());
        items.erase(mid, items.end());
        if (int rc = chain_batch_run(plain, threshold)) return rc;
    }
    hipStream_t st = ex().stream;
    // the longest chains first
    std::vector<int> order(items.size());
    for (size_t k = 0; k < items.size(); ++k) order[k] = (int)k;
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) {
        return items[x].s->dim * items[x].nlanc > items[y].s->dim * items[y].nlanc;
    });
    size_t ncoef = 0, lds = 0;
    for (auto &it : items) ncoef += 2 * (size_t)it.nlanc;
    const size_t nargs = (items.size() * sizeof(WgArgs<double>) + 255) / 256 * 256;
    char *buf = nullptr;
    if (int rc = exec_try(ex(), kSlotChainBatch, nargs + ncoef * 8, (void **)&buf)) return rc;
    double *coef = reinterpret_cast<double *>(buf + nargs);
    std::vector<WgArgs<double>> args;
    for (int k : order) {
        ChainBatchItem &it = items[k];
        const WgShape w = wg_shape(it.s, DMED_FP64);
        if (w.bs == 0) return fail(DMED_EINVAL, "chain batch: sector not taken");
        WgArgs<double> a = wg_args<double>(it.s, w);
        // the shape's columns per lane serve any workgroup of at least its size
        a.v = static_cast<double *>(it.v);
        a.count = a.nlanc = it.nlanc;
        a.thr = threshold;
        a.alpha = coef;
        a.beta = coef + it.nlanc;
        coef += 2 * (size_t)it.nlanc;
        lds = std::max(lds, w.lds);
        args.push_back(a);
    }
    if (int rc = copy_h2d(buf, args.data(), args.size() * sizeof(args[0]))) return rc;
    const auto kern = items[0].s->jterms ? k_chain_wg_batch<true> : k_chain_wg_batch<false>;
    if (int rc = lds_attr_once((const void *)kern)) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)items.size()), dim3(1024), lds, st,
                       reinterpret_cast<const WgArgs<double> *>(buf));
    DMED_HIP(hipGetLastError());
    std::vector<double> h(ncoef);
    DMED_HIP(hipMemcpyAsync(h.data(), buf + nargs, ncoef * 8, hipMemcpyDeviceToHost, st));
    DMED_HIP(hipStreamSynchronize(st));
    const double *c = h.data();
    for (int k : order) {
        ChainBatchItem &it = items[k];
        std::copy(c, c + it.nlanc, it.alpha);
        std::copy(c + it.nlanc, c + 2 * it.nlanc, it.beta);
        c += 2 * it.nlanc;
    }
    return 0;
}

}  // namespace dmed
