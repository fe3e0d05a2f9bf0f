// gf.hip -- Green's functions and susceptibilities of Lanczos chains on the
// device.
//
// add_to_lanczos_gf_normal (build_gf_normal.f90:442-488) diagonalises a
// chain's tridiagonal matrix T (tql2) and sums its poles,
//   G(z) += peso * sum_j Z(1,j)^2 / (z - isign*(lam_j - E)).
// The sum is <e1| (z - isign*(T - E))^-1 |e1>, i.e. the continued fraction of
// the chain's coefficients,
//   G(z) = isign*peso / (t_0),  t_k = s - a_k - b_{k+1}^2 / t_{k+1},
//   s = isign*z + E,
// which needs no diagonalisation: one thread per frequency and chain runs the
// recurrence from the last step to the first.  For Im z != 0 every |t_k| >=
// |Im z|, so the recurrence cannot divide by zero.
//
// Bound by the latency of the recurrence (one division a step); frequencies
// and chains are spread over the chip, so a sum over 4596 frequencies and
// two 200-step chains is one launch of that latency.  On the host the same
// sum took 2.3 ms of tql2 and 0.7 ms of poles for each such chain.  Measured,
// the two Green's-function chains of a state with their sums: 10.0 -> 6.9 ms
// at Ns = 8 (200 steps), 25.3 -> 19.0 ms at Ns = 12 (300 steps); error of
// G(iw) against 64-bit pole sums 1e-14 and 5e-14, both ways alike.
#include <algorithm>
#include <atomic>
#include <cfloat>
#include <cmath>
#include <complex>
#include <cstring>
#include <system_error>
#include <thread>
#include <vector>

#include "dmed_internal.h"
#include "tridiag_device.h"

namespace dmed {

namespace {

// one chain of a sum, as the device reads it
struct CfChain {
    double pr, pi;          // complex weight, isign folded in
    double ei;
    int32_t isign, n, off;  // off: first coefficient pair
    int32_t pad;
};

constexpr int kCfBlock = 64;

// part[chain * nf + i] = 1 / t_0 of the chain at frequency i: i*w_i for
// i < lm, w_i + i*eps after.  AB holds the pairs (a_k, b_{k+1}^2).
__global__ void __launch_bounds__(kCfBlock) k_gf_cf(const CfChain *__restrict__ ch,
                                                    const double2 *__restrict__ AB,
                                                    const double *__restrict__ w, int lm, int nf,
                                                    double eps, double2 *__restrict__ part)
{
    const int i = blockIdx.x * kCfBlock + threadIdx.x;
    if (i >= nf) return;
    const CfChain c = ch[blockIdx.y];
    const double sg = (double)c.isign;
    const double x = (i < lm ? 0.0 : sg * w[i]) + c.ei, y = sg * (i < lm ? w[i] : eps);
    // t = s - a_k - b_{k+1}^2 / t, b_n = 0
    double tr = 1.0, ti = 0.0;
    for (int k = c.n - 1; k >= 0; --k) {
        const double2 ab = AB[c.off + k];
        const double q = ab.y / (tr * tr + ti * ti);
        tr = x - ab.x - q * tr;
        ti = y + q * ti;
    }
    const double q = 1.0 / (tr * tr + ti * ti);
    part[(int64_t)blockIdx.y * nf + i] = make_double2(tr * q, -ti * q);
}

// out[i] = sum over the chains, in order, of weight * part
__global__ void __launch_bounds__(kCfBlock) k_gf_sum(const CfChain *__restrict__ ch, int nch,
                                                     const double2 *__restrict__ part, int nf,
                                                     double2 *__restrict__ out, int first)
{
    const int i = blockIdx.x * kCfBlock + threadIdx.x;
    if (i >= nf) return;
    double2 s = first ? make_double2(0.0, 0.0) : out[i];
    for (int c = 0; c < nch; ++c) {
        const double2 p = part[(int64_t)c * nf + i];
        s.x += ch[c].pr * p.x - ch[c].pi * p.y;
        s.y += ch[c].pr * p.y + ch[c].pi * p.x;
    }
    out[i] = s;
}

// chains of one launch: bounds the partial results to kCfBatch*nf*16 bytes
constexpr int kCfBatch = 64;

int gf_sum_device(const std::vector<GfTerm> &terms, const double *wm, int lm, const double *wr,
                  int lr, double eps, double *g)
{
    const int nf = lm + lr, nt = (int)terms.size();
    hipStream_t st = ex().stream;
    // one upload: frequencies, chain headers, coefficient pairs
    size_t nab = 0;
    for (const GfTerm &t : terms) nab += t.n;
    const size_t ofreq = 0, ohdr = ofreq + (((size_t)nf * 8 + 15) & ~(size_t)15);
    const size_t oab = ohdr + (((size_t)nt * sizeof(CfChain) + 15) & ~(size_t)15);
    const size_t nup = oab + nab * 16;
    const size_t oout = nup, opart = oout + (size_t)nf * 16;
    const size_t total = opart + (size_t)std::min(nt, kCfBatch) * nf * 16;
    std::vector<unsigned char> h(nup);
    double *hw = reinterpret_cast<double *>(h.data());
    if (lm) std::copy(wm, wm + lm, hw);
    if (lr) std::copy(wr, wr + lr, hw + lm);
    CfChain *hc = reinterpret_cast<CfChain *>(h.data() + ohdr);
    double *ab = reinterpret_cast<double *>(h.data() + oab);
    int32_t off = 0;
    for (int k = 0; k < nt; ++k) {
        const GfTerm &t = terms[k];
        hc[k] = CfChain{t.isign * t.pr, t.isign * t.pi, t.ei, t.isign, t.n, off, 0};
        for (int i = 0; i < t.n; ++i, ++off) {
            const double b = i + 1 < t.n ? t.beta[i + 1] : 0.0;
            ab[2 * (size_t)off] = t.alpha[i];
            ab[2 * (size_t)off + 1] = b * b;
        }
    }
    unsigned char *d = nullptr;
    if (int rc = exec_try(ex(), kSlotGf, total, (void **)&d)) return rc;
    DMED_HIP(hipMemcpyAsync(d, h.data(), nup, hipMemcpyHostToDevice, st));
    const CfChain *dc = reinterpret_cast<const CfChain *>(d + ohdr);
    double2 *dout = reinterpret_cast<double2 *>(d + oout);
    double2 *dpart = reinterpret_cast<double2 *>(d + opart);
    const unsigned gx = (unsigned)((nf + kCfBlock - 1) / kCfBlock);
    for (int c0 = 0; c0 < nt; c0 += kCfBatch) {
        const int nc = std::min(kCfBatch, nt - c0);
        hipLaunchKernelGGL(k_gf_cf, dim3(gx, (unsigned)nc), dim3(kCfBlock), 0, st, dc + c0,
                           reinterpret_cast<const double2 *>(d + oab),
                           reinterpret_cast<const double *>(d + ofreq), lm, nf, eps, dpart);
        hipLaunchKernelGGL(k_gf_sum, dim3(gx), dim3(kCfBlock), 0, st, dc + c0, nc, dpart, nf, dout,
                           c0 == 0 ? 1 : 0);
    }
    DMED_HIP(hipGetLastError());
    DMED_HIP(hipMemcpyAsync(g, dout, (size_t)nf * 16, hipMemcpyDeviceToHost, st));
    DMED_HIP(hipStreamSynchronize(st));
    return 0;
}

// poles on the host (tql2): the general form
int gf_sum_host(const std::vector<GfTerm> &terms, const double *wm, int lm, const double *wr,
                int lr, double eps, double *g)
{
    std::vector<double> d, e, z, t(2 * (size_t)(lm + lr));
    std::fill(g, g + t.size(), 0.0);
    for (const GfTerm &c : terms) {
        d.assign(c.alpha, c.alpha + c.n);
        e.assign(c.n, 0.0);
        z.assign(c.n, 0.0);
        for (int i = 1; i < c.n; ++i) e[i] = c.beta[i];
        if (tql2_first_row(c.n, d.data(), e.data(), z.data()))
            return fail(DMED_ENOCONV, "tql2 did not converge");
        for (auto &x : z) x *= x;
        if (c.pi == 0.0) {
            gf_add_poles(c.pr, c.ei, d.data(), z.data(), c.n, c.isign, wm, lm, wr, lr, eps, g,
                         g + 2 * (size_t)lm);
            continue;
        }
        std::fill(t.begin(), t.end(), 0.0);
        gf_add_poles(1.0, c.ei, d.data(), z.data(), c.n, c.isign, wm, lm, wr, lr, eps, t.data(),
                     t.data() + 2 * (size_t)lm);
        for (int i = 0; i < lm + lr; ++i) {
            g[2 * i] += c.pr * t[2 * i] - c.pi * t[2 * i + 1];
            g[2 * i + 1] += c.pr * t[2 * i + 1] + c.pi * t[2 * i];
        }
    }
    return 0;
}

// ------------------------------------------------------- susceptibilities
// The susceptibility sums (build_chi_spin.f90:186-250, build_chi_dens.f90:
// 505-733) weigh every pole with exp(-beta dE) and need chi(tau), so they
// take the poles themselves.  k_chain_poles finds those of many chains (the
// implicit QL iteration of tql2_first_row, one wave per chain, all chains of a
// solve in one launch), the host those of a few; k_chi_prep turns them into the factors that do not depend on
// the frequency, k_chi_term sums one term's poles at one point per thread
// and k_chi_sum adds a target's terms in order.
//
// The QL recurrence is serial (about 0.8 n^2 rotations, each one reciprocal
// square root after the other), so a chain costs its latency, 190 n^2 ns here
// and 37 n^2 ns on the host (200 steps: 7.7 and 1.5 ms): the launch pays from
// about 40 chains on eight host threads, or five on one (chi_route).
// Measured on a two-orbital Ns = 8 solve at beta = 100 with both
// susceptibilities (40 to 200 chains): 374 -> 213 ms.

// n poles of one chain
struct PoleChain {
    int32_t n, off;
};

// Eigenvalues (not sorted) and squared first eigenvector components of the
// chains' tridiagonal matrices, one wave per block; AB holds (a_k, b_k), b_0
// unused.  status: 0, or 1 if an
// eigenvalue took more than 30 iterations.
__global__ void __launch_bounds__(64) k_chain_poles(const PoleChain *__restrict__ ch,
                                                    const double2 *__restrict__ AB,
                                                    double2 *__restrict__ poles,
                                                    int32_t *__restrict__ status)
{
    extern __shared__ double smem[];
    __shared__ double sink[kQlSink];
    const PoleChain c0 = ch[blockIdx.x];
    const int n = c0.n, lane = threadIdx.x;
    double *d = smem, *e = smem + n, *z = smem + 2 * n;
    for (int i = lane; i < n; i += 64) {
        const double2 ab = AB[c0.off + i];
        d[i] = ab.x;
        if (i > 0) e[i - 1] = ab.y;
        z[i] = i == 0 ? 1.0 : 0.0;
    }
    if (lane == 0) e[n - 1] = 0.0;
    __syncthreads();
    const double sc = ql_scale(d, e, n);
    for (int i = lane; i < n; i += 64) {
        d[i] *= sc;
        e[i] *= sc;
    }
    __syncthreads();
    double f = 0.0, tst1 = 0.0;
    bool bad = false;
    for (int l = 0; l < n && !bad; ++l) {
        tst1 = fmax(tst1, fabs(d[l]) + fabs(e[l]));
        const int m = ql_find(e, n, l, tst1);
        for (int iter = 0; m != l; ++iter) {
            if (iter >= 30) {
                bad = true;
                break;
            }
            const double el = ql_iterate<false>(d, e, n, l, m, f, nullptr, nullptr, z, sink);
            if (!(tst1 + el > tst1)) break;
        }
        wave_lds_fence();
        if (lane == 0) d[l] += f;
        wave_lds_fence();
    }
    for (int i = lane; i < n; i += 64) poles[c0.off + i] = make_double2(d[i] / sc, z[i] * z[i]);
    if (lane == 0) status[blockIdx.x] = bad ? 1 : 0;
}

// one term of a susceptibility sum, as the device reads it
struct ChiDev {
    double pr, pi, bz, ei;
    int32_t isign, iv0, n, off;     // off: the chain's first pole
    int32_t poff, target;           // poff: first prepared factor
};

// frequency-independent factors of a term's poles:
// x: signed dE, y: weight*num of the iv and real axes, z: weight, w: weight*f
// of the iv = 0 point
__global__ void __launch_bounds__(64) k_chi_prep(const ChiDev *__restrict__ t,
                                                 const double2 *__restrict__ poles, double beta,
                                                 double4 *__restrict__ fac)
{
    const ChiDev c = t[blockIdx.y];
    const int j = blockIdx.x * 64 + threadIdx.x;
    if (j >= c.n) return;
    const double2 p = poles[c.off + j];
    const double de = p.x - c.ei, ww = p.y * c.bz, ex = exp(-beta * de);
    const double num = c.isign > 0 ? ex - 1.0 : 1.0 - ex;
    fac[c.poff + j] = make_double4(c.isign > 0 ? de : -de, ww * num, ww,
                                   ww * (beta * de < 1e-1 ? beta : (1.0 - ex) / de));
}

// part[term * np + i]: the term's sum at point i (iv, then tau, then real
// axis), before its complex weight
__global__ void __launch_bounds__(64) k_chi_term(const ChiDev *__restrict__ t,
                                                 const double4 *__restrict__ fac,
                                                 const double *__restrict__ x, int nv, int nt,
                                                 int np, double beta, double eps,
                                                 double2 *__restrict__ part)
{
    const int i = blockIdx.x * 64 + threadIdx.x;
    if (i >= np) return;
    const ChiDev c = t[blockIdx.y];
    const double4 *f = fac + c.poff;
    const double xi = x[i];
    double re = 0.0, im = 0.0;
    if (i < nv) {
        if (i == 0) {
            for (int j = 0; j < c.n; ++j) re += f[j].w;
            re *= c.iv0;
        } else {
            for (int j = 0; j < c.n; ++j) {
                // num/(i vm - sde) = num*(-sde - i vm)/(sde^2 + vm^2)
                const double sde = f[j].x, g = f[j].y / (sde * sde + xi * xi);
                re -= sde * g;
                im -= xi * g;
            }
        }
    } else if (i < nv + nt) {
        // signed dE is -dE on the isign = -1 branch: exp(-(beta - tau)*dE)
        for (int j = 0; j < c.n; ++j)
            re += f[j].z * (c.isign > 0 ? exp(-xi * f[j].x) : exp((beta - xi) * f[j].x));
    } else {
        for (int j = 0; j < c.n; ++j) {
            const double y = xi - f[j].x, g = f[j].y / (y * y + eps * eps);
            re += y * g;
            im -= eps * g;
        }
    }
    part[(int64_t)blockIdx.y * np + i] = make_double2(re, im);
}

// out[target * np + i] += the target's terms [c0, c1) in order, with their
// weights (tau: their real part)
__global__ void __launch_bounds__(64) k_chi_sum(const ChiDev *__restrict__ t, int c0, int c1,
                                                const int32_t *__restrict__ toff,
                                                const double2 *__restrict__ part, int nv, int nt,
                                                int np, double2 *__restrict__ out)
{
    const int i = blockIdx.x * 64 + threadIdx.x;
    if (i >= np) return;
    const int q = blockIdx.y;
    double2 s = c0 == 0 ? make_double2(0.0, 0.0) : out[(int64_t)q * np + i];
    for (int c = max(c0, toff[q]); c < min(c1, toff[q + 1]); ++c) {
        const double2 p = part[(int64_t)(c - c0) * np + i];
        s.x += t[c].pr * p.x - t[c].pi * p.y;
        s.y += t[c].pr * p.y + t[c].pi * p.x;
    }
    out[(int64_t)q * np + i] = s;
}

// terms of one launch: bounds the partial results to kChiBatch*np*16 bytes
constexpr int kChiBatch = 256;

// poles of the chains on nthread host threads, the longest first: over the
// coefficient pairs, as k_chain_poles would leave them
int chi_poles_host(const std::vector<PoleChain> &ch, int nthread, double *ab)
{
    std::vector<int> order(ch.size());
    for (size_t k = 0; k < ch.size(); ++k) order[k] = (int)k;
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return ch[x].n > ch[y].n; });
    std::atomic<size_t> next(0);
    std::atomic<int> bad(0);
    auto work = [&]() {
        std::vector<double> d, e, z;
        for (size_t k; (k = next.fetch_add(1)) < order.size();) {
            const PoleChain c = ch[order[k]];
            double *p = ab + 2 * (size_t)c.off;
            d.resize(c.n);
            e.resize(c.n);
            z.resize(c.n);
            for (int i = 0; i < c.n; ++i) {
                d[i] = p[2 * i];
                e[i] = p[2 * i + 1];
            }
            if (tql2_first_row(c.n, d.data(), e.data(), z.data())) bad = 1;
            for (int i = 0; i < c.n; ++i) {
                p[2 * i] = d[i];
                p[2 * i + 1] = z[i] * z[i];
            }
        }
    };
    std::vector<std::thread> th;
    try {
        for (int t = 1; t < nthread; ++t) th.emplace_back(work);
    } catch (const std::system_error &) {
        // fewer threads than asked for
    }
    work();
    for (auto &t : th) t.join();
    return bad ? fail(DMED_ENOCONV, "tql2 did not converge") : 0;
}

// terms sorted by target; nthread > 0: poles on that many host threads
int chi_sum_device(const std::vector<ChiTerm> &terms, int ntarget, double beta, const ChiGrid &g,
                   double *out, int nthread)
{
    hipStream_t st = ex().stream;
    const int np = g.nv + g.nt + g.lr, nterm = (int)terms.size();
    // a chain's isign = +1 and -1 terms are neighbours: its poles are found once
    std::vector<PoleChain> ch;
    std::vector<const double *> src;
    std::vector<ChiDev> dev;
    std::vector<int32_t> toff(ntarget + 1, 0);
    std::vector<double> ab;
    int32_t poff = 0, nmax = 1;
    for (const ChiTerm &t : terms) {
        if (src.empty() || src.back() != t.alpha || ch.back().n != t.n) {
            src.push_back(t.alpha);
            ch.push_back(PoleChain{t.n, (int32_t)(ab.size() / 2)});
            for (int i = 0; i < t.n; ++i) {
                ab.push_back(t.alpha[i]);
                ab.push_back(i ? t.beta[i] : 0.0);
            }
        }
        dev.push_back(ChiDev{t.pr, t.pi, t.peso_bz, t.ei, t.isign, t.iv0_sign, t.n, ch.back().off, poff,
                             t.target});
        poff += t.n;
        nmax = std::max(nmax, (int32_t)t.n);
        ++toff[t.target + 1];
    }
    for (int q = 0; q < ntarget; ++q) toff[q + 1] += toff[q];
    if (nthread > 0)
        if (int rc = chi_poles_host(ch, nthread, ab.data())) return rc;
    const size_t nch = ch.size();
    auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
    const size_t ox = 0, och = ox + up((size_t)np * 8), odev = och + up(nch * sizeof(PoleChain));
    const size_t otoff = odev + up((size_t)nterm * sizeof(ChiDev));
    const size_t oab = otoff + up(toff.size() * 4), nup = oab + up(ab.size() * 8);
    const size_t opole = nup, ofac = opole + up(ab.size() * 8), ost = ofac + up((size_t)poff * 32);
    const size_t oout = ost + up(nch * 4), opart = oout + up((size_t)ntarget * np * 16);
    const size_t total = opart + (size_t)std::min(nterm, kChiBatch) * np * 16;
    std::vector<unsigned char> h(nup);
    double *hx = reinterpret_cast<double *>(h.data());
    if (g.nv) std::copy(g.vm, g.vm + g.nv, hx);
    if (g.nt) std::copy(g.tau, g.tau + g.nt, hx + g.nv);
    if (g.lr) std::copy(g.wr, g.wr + g.lr, hx + g.nv + g.nt);
    std::memcpy(h.data() + och, ch.data(), nch * sizeof(PoleChain));
    std::memcpy(h.data() + odev, dev.data(), dev.size() * sizeof(ChiDev));
    std::memcpy(h.data() + otoff, toff.data(), toff.size() * 4);
    std::memcpy(h.data() + oab, ab.data(), ab.size() * 8);
    unsigned char *d = nullptr;
    if (int rc = exec_try(ex(), kSlotGf, total, (void **)&d)) return rc;
    DMED_HIP(hipMemcpyAsync(d, h.data(), nup, hipMemcpyHostToDevice, st));
    const ChiDev *dt = reinterpret_cast<const ChiDev *>(d + odev);
    double2 *dpole = reinterpret_cast<double2 *>(d + (nthread > 0 ? oab : opole));
    double4 *dfac = reinterpret_cast<double4 *>(d + ofac);
    double2 *dout = reinterpret_cast<double2 *>(d + oout);
    double2 *dpart = reinterpret_cast<double2 *>(d + opart);
    if (nthread == 0)
        hipLaunchKernelGGL(k_chain_poles, dim3((unsigned)nch), dim3(64), (size_t)nmax * 24, st,
                           reinterpret_cast<const PoleChain *>(d + och),
                           reinterpret_cast<const double2 *>(d + oab), dpole,
                           reinterpret_cast<int32_t *>(d + ost));
    const unsigned gx = (unsigned)((np + 63) / 64);
    for (int c0 = 0; c0 < nterm; c0 += kChiBatch) {
        const int nc = std::min(kChiBatch, nterm - c0);
        hipLaunchKernelGGL(k_chi_prep, dim3((unsigned)((nmax + 63) / 64), (unsigned)nc), dim3(64), 0,
                           st, dt + c0, dpole, beta, dfac);
        hipLaunchKernelGGL(k_chi_term, dim3(gx, (unsigned)nc), dim3(64), 0, st, dt + c0, dfac,
                           reinterpret_cast<const double *>(d + ox), g.nv, g.nt, np, beta, g.eps,
                           dpart);
        hipLaunchKernelGGL(k_chi_sum, dim3(gx, (unsigned)ntarget), dim3(64), 0, st, dt, c0, c0 + nc,
                           reinterpret_cast<const int32_t *>(d + otoff), dpart, g.nv, g.nt, np, dout);
    }
    DMED_HIP(hipGetLastError());
    std::vector<int32_t> bad(nch, 0);
    if (nthread == 0)
        DMED_HIP(hipMemcpyAsync(bad.data(), d + ost, nch * 4, hipMemcpyDeviceToHost, st));
    DMED_HIP(hipMemcpyAsync(out, dout, (size_t)ntarget * np * 16, hipMemcpyDeviceToHost, st));
    DMED_HIP(hipStreamSynchronize(st));
    for (int32_t b : bad)
        if (b) return DMED_ENOCONV;
    return 0;
}

int chi_sum_host(const std::vector<ChiTerm> &terms, double beta, const ChiGrid &g, double *out)
{
    const int np = g.nv + g.nt + g.lr;
    std::vector<double> d, e, z, tau(g.nt);
    const double *last = nullptr;
    for (const ChiTerm &t : terms) {
        if (t.alpha != last || (int)d.size() != t.n) {
            d.assign(t.alpha, t.alpha + t.n);
            e.assign(t.n, 0.0);
            z.assign(t.n, 0.0);
            for (int i = 1; i < t.n; ++i) e[i] = t.beta[i];
            if (tql2_first_row(t.n, d.data(), e.data(), z.data()))
                return fail(DMED_ENOCONV, "tql2 did not converge");
            for (auto &x : z) x *= x;
            last = t.alpha;
        }
        double *o = out + 2 * (size_t)t.target * np;
        std::fill(tau.begin(), tau.end(), 0.0);
        chi_add_branch(t.pr, t.pi, t.peso_bz, t.ei, d.data(), z.data(), t.n, t.isign, t.iv0_sign, beta,
                       g.vm, g.nv, g.tau, g.nt, g.wr, g.lr, g.eps, o, tau.data(),
                       o + 2 * (size_t)(g.nv + g.nt));
        for (int i = 0; i < g.nt; ++i) o[2 * (size_t)(g.nv + i)] += tau[i];
    }
    return 0;
}

}  // namespace

// Whether the host form takes over after a device sum returned rc: where its
// buffer could not be had or its pole iteration did not converge.  A HIP error
// goes to the caller.
bool host_may_take(int rc) { return rc == DMED_ENOMEM || rc == DMED_ENOCONV; }

// Whether a sum runs on the device.  The continued fraction needs every point
// off the real axis (1e-100: its square is still a normal number) and finite
// coefficients.  The upload, two launches and the download take 36 us; the
// host takes 50 n^2 ns for the poles of a short chain and 0.5 ns per pole and
// frequency (n = 20: 22 us at 8 frequencies, 27 at 512; n = 10 at 4596: 33).
bool gf_on_device(const std::vector<GfTerm> &terms, const double *wm, int lm, const double *wr, int lr,
                  double eps)
{
    constexpr double kDeviceNs = 36e3;
    double host_ns = 0.0;
    bool ok = ctx().initialized && lm + lr > 0;
    for (const GfTerm &t : terms) {
        host_ns += (50.0 * t.n + 0.5 * ((double)lm + lr)) * t.n;
        for (int i = 0; i < t.n && ok; ++i)
            ok = std::fabs(t.alpha[i]) < 1e100 && (i == 0 || std::fabs(t.beta[i]) < 1e100);
        ok = ok && std::fabs(t.ei) < 1e100 && (t.isign == 1 || t.isign == -1);
    }
    ok = ok && host_ns > kDeviceNs && (lr == 0 || (std::fabs(eps) > 1e-100 && std::fabs(eps) < 1e100));
    for (int i = 0; i < lm && ok; ++i) ok = std::fabs(wm[i]) > 1e-100 && std::fabs(wm[i]) < 1e100;
    for (int i = 0; i < lr && ok; ++i) ok = std::fabs(wr[i]) < 1e100;
    return ok;
}

// g[0..lm) on the Matsubara axis, g[lm..lm+lr) on the real axis, overwritten
// with the sum over the terms
int gf_sum(const std::vector<GfTerm> &terms, const double *wm, int lm, const double *wr, int lr,
           double eps, double *g, bool on_device)
{
    if (on_device) {
        const int rc = gf_sum_device(terms, wm, lm, wr, lr, eps, g);
        if (!host_may_take(rc)) return rc;
    }
    return gf_sum_host(terms, wm, lm, wr, lr, eps, g);
}

// Where a susceptibility sum runs, terms sorted by target: -1 on the host; else
// on the device, with the poles on that many host threads, 0: on the device
// too.  Coefficients that are not finite go to the host.  Measured: a wave
// takes 60 us and 190 n^2 ns for the poles of a chain, the host 37 n^2 ns;
// the sums cost the device 45 us and 0.4 us per pole of the longest chain, and
// the host 0.8 ns per pole of a term and point of the iv and real axes and 2.8
// ns per point of the tau axis.  One chain of 200 steps, 1626 points: 2.05 ms
// on the host alone, 1.55 ms with the sums here, 7.8 ms with the poles here too.
// Threads of a solve's own (sites) take their chains alone.
int chi_route(const std::vector<ChiTerm> &terms, const ChiGrid &g)
{
    constexpr int kMaxSteps = 2048;             // 3 doubles a step in LDS
    static const size_t kThreads = std::min(8u, std::max(1u, std::thread::hardware_concurrency()));
    double nmax = 0.0, sq = 0.0, sum_ns = 0.0;
    size_t nsum = 0, nch = 0;
    const double *last = nullptr;
    bool ok = ctx().initialized && g.nv + g.nt + g.lr > 0;
    for (const ChiTerm &t : terms) {
        nsum += t.n;
        sum_ns += t.n * (0.8 * ((double)g.nv + g.lr) + 2.8 * g.nt);
        if (t.alpha != last) {
            nmax = std::max(nmax, (double)t.n);
            sq += (double)t.n * t.n;
            ++nch;
        }
        last = t.alpha;
        for (int i = 0; i < t.n && ok; ++i)
            ok = std::fabs(t.alpha[i]) < 1e100 && (i == 0 || std::fabs(t.beta[i]) < 1e100);
    }
    if (!ok || nsum >= ((size_t)1 << 24)) return -1;        // 64 B of work space a pole
    // threads where the chains take longer than starting them
    const int nthread = &ex() == &ctx().exec && 37.0 * sq > 300e3 ? (int)std::min(nch, kThreads) : 1;
    const double host_ns = 37.0 * std::max(nmax * nmax, sq / nthread);
    if (nmax <= kMaxSteps && host_ns > 60e3 + 190.0 * nmax * nmax) return 0;
    return sum_ns > 45e3 + 400.0 * nmax ? nthread : -1;
}

// out[target * np + i], np = nv + nt + lr points (iv, tau, real axis),
// interleaved complex (tau: its real part), overwritten with the sums over
// the terms
int chi_sum(std::vector<ChiTerm> terms, int ntarget, double beta, const ChiGrid &g, double *out,
            const int *known_route)
{
    std::fill(out, out + 2 * (size_t)ntarget * (g.nv + g.nt + g.lr), 0.0);
    if (terms.empty()) return 0;
    std::stable_sort(terms.begin(), terms.end(),
                     [](const ChiTerm &a, const ChiTerm &b) { return a.target < b.target; });
    const int route = known_route ? *known_route : chi_route(terms, g);
    if (route >= 0) {
        const int rc = chi_sum_device(terms, ntarget, beta, g, out, route);
        if (!host_may_take(rc)) return rc;
    }
    std::fill(out, out + 2 * (size_t)ntarget * (g.nv + g.nt + g.lr), 0.0);
    return chi_sum_host(terms, beta, g, out);
}

}  // namespace dmed
