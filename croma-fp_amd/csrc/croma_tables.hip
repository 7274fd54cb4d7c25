// Grid-constant kernel tables built on the device: the secondary weights and
// the gamma and neutrino rows from the shared physics header
// (croma_hadronic.h), one table entry per thread; the IC rows from this file's
// own form of the integrand (k_ic_table), eight lanes per entry:
//   secondary-electron weights fqe_t[jp][je]   fp_shared_core.c:1453-1506 (QeKernel_BB05, HADRONIC.c:436-498)
//   gamma / neutrino / IC kernel tables [k][j]  fp_shared_core.c:1724-1804 (prepare_*_kernel_flat),
//                                              HADRONIC.c:139-289, FP_Coef.c:553-582
// Every entry is an independent FP64 quadrature of 50..400 nodes (pow /
// log10 / exp per node), so the tables are FP64-VALU bound;
// threads of a wave walk consecutive columns so each store is coalesced.
#include <hip/hip_runtime.h>

#include "croma_hadronic.h"
#include "croma_kernels.h"

namespace {

constexpr int kTabBlock = 128;

// vals[jp][je] = QeKernel(E_e[je], p[jp]) * beta_p[jp], NaN -> 0
// (fp_shared_core.c:1464-1471).
__global__ void __launch_bounds__(kTabBlock) k_fqe_vals(int n, const double *__restrict__ e_energy,
                                                         const double *__restrict__ pp,
                                                         const double *__restrict__ beta_p, double *vals)
{
    const int je = blockIdx.x * kTabBlock + threadIdx.x;
    const int jp = blockIdx.y;
    if (je >= n) return;
    double v = chk_qe_kernel(e_energy[je], pp[jp]) * beta_p[jp];
    if (isnan(v)) v = 0.0;
    vals[(size_t)jp * n + je] = v;
}

// Per electron bin je: jp0 = 1 + the last proton bin whose value is below
// 1e-80 (at least 1), then the trapezoid weights over proton bins jp0-1..n-1
// replace the values in place (fp_shared_core.c:1473-1503).  np_min[je] is
// jp0 - 1, or n when no proton bin contributes.
__global__ void __launch_bounds__(kTabBlock) k_fqe_weights(int n, const double *__restrict__ pdp, double *fqe,
                                                            int *np_min)
{
    const int je = blockIdx.x * kTabBlock + threadIdx.x;
    if (je >= n) return;
    int npmin = 1;
    for (int jp = 1; jp < n; jp++)
        if (fqe[(size_t)jp * n + je] < 1.0e-80) npmin = jp;
    const int jp0 = npmin < 1 ? 1 : (npmin > n ? n : npmin);
    for (int jp = 0; jp < n; jp++) {
        const size_t at = (size_t)jp * n + je;
        const double v = fqe[at];
        double w = 0.0;
        if (jp0 < n) {
            if (jp == jp0 - 1) w = 0.5 * v * pdp[jp0];
            else if (jp >= jp0 && jp < n - 1) w = 0.5 * v * (pdp[jp] + pdp[jp + 1]);
            else if (jp == n - 1 && jp >= jp0) w = 0.5 * v * pdp[jp];
        }
        fqe[at] = w;
    }
    np_min[je] = (jp0 < n) ? (jp0 - 1) : n;
}

// out[k][j] for k < nbins on the accumulated log grid a_k = lo + (k+1) d - d
// summed term by term as the reference's loops do (so a_k is bit-identical
// to theirs, fp_shared_core.c:1735-1741); kind 0 gamma(E_k, p_j), 1 neutrino(E_k, p_j).
__global__ void __launch_bounds__(kTabBlock) k_emis_table(int kind, int n, int nbins, double lo, double d,
                                                           const double *__restrict__ mom, double *out)
{
    const int j = blockIdx.x * kTabBlock + threadIdx.x;
    const int k = blockIdx.y;
    if (j >= n || k >= nbins) return;
    double a = lo - d;
    for (int kk = 0; kk <= k; kk++) a += d;
    const double e = pow(10.0, a);
    const double p = mom[j];
    double v;
    if (kind == 0) v = chk_gamma_kernel(e, p);
    else v = chk_nu_kernel(e, p);
    out[(size_t)k * n + j] = v;
}

// Inverse-Compton emissivity table: out[k][j], the emissivity at nu_k of an
// electron of gamma = sqrt(1 + p_j^2) in the CMB at z, by the 400-node
// trapezoid rule over log10 of the photon energy (FP_Coef.c:553-582), a table
// per snapshot's redshift.  Bound: FP64 VALU (a pow, a log and an exp per
// node).  One thread per entry left one wave per CU with 400 nodes in a row
// (635 us for 64 x 256 entries); here eight lanes share an entry, 50 nodes
// each, leave their trapezoid terms in LDS and the first of them adds the 400
// terms in the serial order (238 us, the same bits).  The integrand's squares
// are products and its constants are formed once, where pow calls took half of
// the 720 instructions of a node (148 us).
__device__ __forceinline__ double ict_kernel(double eps0, double gamma, double eps)
{
#pragma clang fp contract(off)
    const double re = 2.82e-13;
    const double kappa = eps / (4.0 * eps0 * gamma * (gamma - eps));
    if (kappa <= 0.0) return 0.0;
    const double q = 4.0 * eps0 * kappa * gamma;
    const double C = 2.0 * kappa * log(kappa) + (1.0 + 2.0 * kappa) * (1.0 - kappa) +
                     q * q / (2.0 * (1.0 + 4.0 * eps0 * gamma * kappa)) * (1.0 - kappa);
    return 2.0 * CHK_PI * re * re * CHK_C / (gamma * gamma * eps0) * C;
}

// pre = 8 pi c^3 (m_e / h)^3, kt = k T_cmb
__device__ __forceinline__ double ict_cmb_n(double eps, double pre, double kt)
{
#pragma clang fp contract(off)
    const double meg = 9.11e-28, tiny = 1.0e-40;
    const double x = eps * meg * CHK_C * CHK_C / kt;
    if (x > 90.0 * log(10.0)) return 0.0;
    const double em1 = exp(x) - 1.0;
    if (em1 < tiny) return pre * eps / (meg * CHK_C * CHK_C * (1.0 + 0.5 * x + x / 6.0) / kt);
    return pre * (eps * eps) / em1;
}

constexpr int kIcLanes = 8, kIcNodes = 400, kIcRun = kIcNodes / kIcLanes, kIcGroups = 64 / kIcLanes;

__global__ void __launch_bounds__(64) k_ic_table(int n, int nbins, double lo, double d, double z,
                                                 const double *__restrict__ mom, double *out)
{
    CHK_NOCONTRACT
    __shared__ double s_t[kIcGroups][kIcNodes + 1];
    const int g = threadIdx.x / kIcLanes, c = threadIdx.x % kIcLanes;
    const int j = blockIdx.x * kIcGroups + g, k = blockIdx.y;
    const double meg = 9.11e-28, cl = 3.0e+10;
    const double r = meg / CHK_H, pre = 8.0 * CHK_PI * CHK_C * CHK_C * CHK_C * (r * r * r);
    const double kt = 1.38e-16 * (2.757 * (1.0 + z));
    double ak = lo - d;
    for (int kk = 0; kk <= k; kk++) ak += d;
    const double nu = pow(10.0, ak);
    const double eps = CHK_H * nu / (meg * cl * cl);
    if (j < n) {
        const double p = mom[j], gamma = sqrt(1.0 + p * p);
        double e0max = eps, e0min = eps / (4.0 * gamma * (gamma - eps));
        if (e0min < 0) e0min = eps / (gamma * gamma);
        const double da = (log10(e0max) - log10(e0min)) / (double)kIcNodes;
        double a = log10(e0min);
        for (int i = 0; i < c * kIcRun; i++) a = a + da;
        double e0n = pow(10.0, a), Cn = ict_kernel(e0n, gamma, eps), nn = ict_cmb_n(e0n, pre, kt);
        for (int i = c * kIcRun; i < (c + 1) * kIcRun; i++) {
            const double e0 = e0n, C = Cn, n0 = nn;
            a = a + da;
            e0n = pow(10.0, a);
            nn = ict_cmb_n(e0n, pre, kt);
            Cn = ict_kernel(e0n, gamma, eps);
            s_t[g][i] = 0.5 * (C * n0 + Cn * nn) * (e0n - e0);
        }
    }
    __syncthreads();
    if (j < n && c == 0) {
        double sum = 0.0;
        for (int i = 0; i < kIcNodes; i++) sum = sum + s_t[g][i];
        out[(size_t)k * n + j] = CHK_H * eps * sum / (4.0 * CHK_PI);
    }
}

}  // namespace

extern "C" int ck_secondary_weights(int n, const double *e_energy, const double *pp, const double *beta_p,
                                    const double *pdp, double *fqe_t, int *np_min, void *stream)
{
    if (n <= 0 || n > 65535) return 1;
    const hipStream_t st = (hipStream_t)stream;
    const unsigned gx = (unsigned)((n + kTabBlock - 1) / kTabBlock);
    hipLaunchKernelGGL(k_fqe_vals, dim3(gx, (unsigned)n), dim3(kTabBlock), 0, st, n, e_energy, pp, beta_p, fqe_t);
    hipLaunchKernelGGL(k_fqe_weights, dim3(gx), dim3(kTabBlock), 0, st, n, pdp, fqe_t, np_min);
    return hipGetLastError() != hipSuccess;
}

extern "C" int ck_emission_kernel_table(int kind, int n, int nbins, double lo, double hi, double z,
                                        const double *mom, double *out, void *stream)
{
    if (n <= 0 || nbins <= 0 || nbins > 65535 || kind < 0 || kind > 2) return 1;
    const unsigned gx = (unsigned)((n + kTabBlock - 1) / kTabBlock);
    if (kind == 2) {
        hipLaunchKernelGGL(k_ic_table, dim3((unsigned)((n + kIcGroups - 1) / kIcGroups), (unsigned)nbins), dim3(64), 0,
                           (hipStream_t)stream, n, nbins, lo, (hi - lo) / (double)nbins, z, mom, out);
        return hipGetLastError() != hipSuccess;
    }
    hipLaunchKernelGGL(k_emis_table, dim3(gx, (unsigned)nbins), dim3(kTabBlock), 0, (hipStream_t)stream, kind, n,
                       nbins, lo, (hi - lo) / (double)nbins, mom, out);
    return hipGetLastError() != hipSuccess;
}
