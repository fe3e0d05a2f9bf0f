// gf.hip -- Green's functions of Lanczos chains on the device.
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
#include <cfloat>
#include <cmath>
#include <complex>
#include <cstring>
#include <vector>

#include "dmed_internal.h"

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
    if (int rc = exec_buf(ex(), kSlotGf, total, (void **)&d)) return rc;
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

}  // namespace

// g[0..lm) on the Matsubara axis, g[lm..lm+lr) on the real axis, overwritten
// with the sum over the terms.  The continued fraction needs every point off
// the real axis (1e-100: its square is still a normal number) and finite
// coefficients.  Chains under kCfMin steps stay on the host: their poles cost
// it 10-20 us there, less than the upload, the two launches and the download.
int gf_sum(const std::vector<GfTerm> &terms, const double *wm, int lm, const double *wr, int lr,
           double eps, double *g)
{
    constexpr int kCfMin = 16;
    int nmax = 0;
    bool ok = ctx().initialized && lm + lr > 0;
    for (const GfTerm &t : terms) {
        nmax = std::max(nmax, t.n);
        for (int i = 0; i < t.n && ok; ++i)
            ok = std::fabs(t.alpha[i]) < 1e100 && (i == 0 || std::fabs(t.beta[i]) < 1e100);
        ok = ok && std::fabs(t.ei) < 1e100 && (t.isign == 1 || t.isign == -1);
    }
    ok = ok && nmax >= kCfMin && (lr == 0 || (std::fabs(eps) > 1e-100 && std::fabs(eps) < 1e100));
    for (int i = 0; i < lm && ok; ++i) ok = std::fabs(wm[i]) > 1e-100 && std::fabs(wm[i]) < 1e100;
    for (int i = 0; i < lr && ok; ++i) ok = std::fabs(wr[i]) < 1e100;
    if (ok && gf_sum_device(terms, wm, lm, wr, lr, eps, g) == 0) return 0;
    return gf_sum_host(terms, wm, lm, wr, lr, eps, g);
}

}  // namespace dmed
