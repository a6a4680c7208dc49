// spectra.hip -- kinetic-energy spectrum of the live velocity field.
//
// The reference leaves spectra to post-processing on the dumps
// (python_utilities/plot_fields.py:116-151, a 1-D FFT of one profile) and
// the dissipation to post/compute_diss.  Here the 3-D shell spectrum
//   E(k) = 1/2 sum_{k - 1/2 <= |m| < k + 1/2} (|u^(m)|^2 + |v^(m)|^2 + |w^(m)|^2) / N^2,
// N = n^3, is computed on the device with the context's own R2C FFT (in the
// Poisson precision), so that sum_k E(k) is the kinetic energy
// 1/2 <u^2 + v^2 + w^2> of mhit_diag.  Each half-spectrum mode with
// 0 < kx < n/2 stands for itself and its Hermitian partner (weight 2); the
// kx = 0 and kx = n/2 (Nyquist) modes count once.  The spectrum buffer is
// scratch between steps.
#include "fft.hpp"
#include "internal.hpp"

#include <algorithm>
#include <cmath>
#include <mutex>
#include <string>

namespace mhit {
int sync_scalars_public(mhit_ctx* c);

int shells_used(int n) { return (int)std::floor(std::sqrt(3.0) * (n / 2) + 0.5) + 1; }

// Two workgroups of eight waves per CU at most.
int spectrum_blocks(int n) { return std::min(512, div_up((long long)n * n * div_up(n / 2, 64), 8)); }
}  // namespace mhit

using namespace mhit;

namespace {

__device__ __forceinline__ int signed_wavenumber(int m, int n) { return m <= n / 2 ? m : m - n; }

// Shell sums of one velocity component, without atomics.  A wave takes 64
// consecutive kx of a (ky, kz) row at a time.  |k| grows along a row, so the
// modes of one shell sit in consecutive lanes: a segmented scan over the
// wave leaves each shell's sum in the last lane of its run, which adds it to
// the wave's own bins in LDS (no two of those lanes share a shell); lane 0
// then adds the row's Nyquist mode.  The workgroup's sums go to
// parts[workgroup][shell] and k_shell_sum adds those up in a fixed order,
// so the result is the same from call to call.
// Bound by reading the spectrum once, the next 64 modes in flight while the
// current ones are binned.  The earlier form, a workgroup per row with an
// LDS and a device-wide FP64 atomic per shell, spent 1.10 ms on the 8.4
// million device-wide atomics of a 256^3 box (FP64 transform); this one
// takes 0.061 ms (2.2 TB/s; the scan's lane exchanges are the rest).
// The k = 0 shell holds the k = 0 mode alone: the square of the component's
// mean, from the stored sum less the deferred mean removal (component f).
constexpr int kBinWaves = 8;

template <typename V>
__global__ __launch_bounds__(64 * kBinWaves)
void k_shell_bins(const V* __restrict__ spec, const V* __restrict__ nyq, int n, const DevScalars* __restrict__ S,
                  int f, double* __restrict__ parts, int nbins) {
    extern __shared__ double sb[];   // [wave][shell]
    for (int b = threadIdx.x; b < kBinWaves * nbins; b += blockDim.x) sb[b] = 0.0;
    __syncthreads();
    const int h = n / 2, nc = (h + 63) / 64, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int total = n * n * nc, stride = gridDim.x * kBinWaves;
    const double cells = (double)n * n * n, scale = 0.5 / (cells * cells);
    // the wave's bins are read and written in program order by it alone
    volatile double* bins = sb + (size_t)w * nbins;
    auto load = [&](int it, V& c, V& cn) {
        if (it >= total) return;
        const int row = it / nc, k0 = (it - row * nc) * 64;
        if (k0 + lane < h) c = spec[(size_t)row * h + k0 + lane];
        if (k0 == 0 && lane == 0) cn = nyq[row];
    };
    auto energy = [&](const V& c, double weight) {
        const double re = (double)c.x, im = (double)c.y;
        return weight * scale * (re * re + im * im);
    };
    V c{}, cn{}, d{}, dn{};
    load(blockIdx.x * kBinWaves + w, c, cn);
    for (int it = blockIdx.x * kBinWaves + w; it < total; it += stride) {
        load(it + stride, d, dn);
        const int row = it / nc, k0 = (it - row * nc) * 64, kx = k0 + lane;
        const int sy = signed_wavenumber(row % n, n), sz = signed_wavenumber(row / n, n);
        const double kyz2 = (double)sy * sy + (double)sz * sz;
        int b = -1 - lane;   // past the row: a run of its own, not stored
        double e = 0.0;
        if (kx < h) {
            e = energy(c, kx == 0 ? 1.0 : 2.0);
            if (row == 0 && kx == 0) {
                const double m = (double)c.x / cells - S->mean[f];
                e = 0.5 * m * m;
            }
            b = (int)floor(sqrt((double)kx * kx + kyz2) + 0.5);
        }
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const double t = __shfl_up(e, o, 64);
            const int bt = __shfl_up(b, o, 64);
            if (lane >= o && bt == b) e += t;
        }
        const int next = __shfl_down(b, 1, 64);
        if ((lane == 63 || next != b) && b >= 0 && b < nbins) bins[b] = bins[b] + e;
        if (k0 == 0 && lane == 0) {
            const int bn = (int)floor(sqrt((double)h * h + kyz2) + 0.5);
            if (bn < nbins) bins[bn] = bins[bn] + energy(cn, 1.0);
        }
        c = d;
        cn = dn;
    }
    __syncthreads();
    for (int b = threadIdx.x; b < nbins; b += blockDim.x) {
        double s = 0.0;
        for (int v = 0; v < kBinWaves; v++) s += sb[(size_t)v * nbins + b];
        parts[(size_t)blockIdx.x * nbins + b] = s;
    }
}

// bins[b] (+)= the sum of parts[.][b]; a wave per shell
__global__ __launch_bounds__(64)
void k_shell_sum(const double* __restrict__ parts, int nparts, int nbins, bool add, double* __restrict__ bins) {
    const int b = blockIdx.x;
    double s = 0.0;
    for (int p = threadIdx.x; p < nparts; p += 64) s += parts[(size_t)p * nbins + b];
    s = wave_sum(s);
    if (threadIdx.x == 0) bins[b] = add ? bins[b] + s : s;
}

// The spectrum with its shell sums in bins[0, min(nbins, shells)) (device
// memory the caller provides); E is written directly, no host staging.
int spectrum_into(mhit_ctx* c, int32_t nbins, double* E, int32_t* nshells, double* bins) {
    const int n = c->n;
    const int used = shells_used(n);
    if (nshells) *nshells = used;
    const int nb = nbins < used ? nbins : used;
    int rc = MHIT_OK;
    const int blocks = spectrum_blocks(n);   // workgroup sums in the diagnostics' partials
    hipError_t err = hipSuccess;
    double* fields[3] = {c->u, c->v, c->w};
    for (int f = 0; f < 3 && err == hipSuccess && rc == MHIT_OK; f++) {
        if ((rc = fft_r2c_dev(c, fields[f]))) break;
        const size_t lds = (size_t)kBinWaves * nb * sizeof(double);
        if (c->fp32)
            k_shell_bins<float2><<<blocks, 64 * kBinWaves, lds, c->stream>>>(
                (const float2*)c->spec, (const float2*)c->nyq, n, c->S, f, c->dpartials, nb);
        else
            k_shell_bins<double2><<<blocks, 64 * kBinWaves, lds, c->stream>>>(
                (const double2*)c->spec, (const double2*)c->nyq, n, c->S, f, c->dpartials, nb);
        k_shell_sum<<<nb, 64, 0, c->stream>>>(c->dpartials, blocks, nb, f > 0, bins);
        err = hipGetLastError();
    }
    if (err == hipSuccess && rc == MHIT_OK)
        err = hipMemcpyAsync(E, bins, (size_t)nb * sizeof(double), hipMemcpyDeviceToHost, c->stream);
    if (err == hipSuccess && rc == MHIT_OK) err = hipStreamSynchronize(c->stream);
    if (rc) return rc;
    MHIT_HIP_TRY(err);
    for (int b = nb; b < nbins; b++) E[b] = 0.0;
    return MHIT_OK;
}

int spectrum_check(mhit_ctx* c, int32_t nbins, double* E) {
    if (!c || nbins <= 0 || !E) { set_error("bad arguments"); return MHIT_ERR_ARG; }
    int rc;
    if ((rc = sync_scalars_public(c))) return rc;
    if (c->S_host.halted) { set_error("stopped: cou > 7"); return MHIT_ERR_CFL; }
    return MHIT_OK;
}

// Shell sums of mhit_energy_spectrum_noalloc: one array per device, held
// until the process ends, shared by every call on that device (calls that
// overlap on one device race on it).  Host code never uses the array's
// name as an address: each device's copy is looked up once with
// hipGetSymbolAddress (with that device current) and kept.
constexpr int kScratchBins = MHIT_SPECTRUM_NOALLOC_MAX_BINS;
static __device__ __align__(256) double scratch[kScratchBins];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch[kMaxDevices] = {};

int scratch_on(int device, double** out) {
    if (device < 0 || device >= kMaxDevices) { set_error("device ordinal out of range"); return MHIT_ERR_ARG; }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[device]) {
        int cur = -1;
        MHIT_HIP_TRY(hipGetDevice(&cur));
        if (cur != device) MHIT_HIP_TRY(hipSetDevice(device));
        double* p = nullptr;
        const hipError_t e = hipGetSymbolAddress((void**)&p, HIP_SYMBOL(scratch));
        if (cur != device) MHIT_HIP_TRY(hipSetDevice(cur));
        if (e != hipSuccess || !p) {
            set_error(std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
            return MHIT_ERR_HIP;
        }
        g_scratch[device] = p;
    }
    *out = g_scratch[device];
    return MHIT_OK;
}

}  // namespace

extern "C" {

int mhit_energy_spectrum(mhit_ctx* c, int32_t nbins, double* E, int32_t* nshells) {
    int rc;
    if ((rc = spectrum_check(c, nbins, E))) return rc;
    const int used = shells_used(c->n);
    const int nb = nbins < used ? nbins : used;
    double* bins = nullptr;
    MHIT_HIP_TRY(hipMalloc((void**)&bins, (size_t)nb * sizeof(double)));
    rc = spectrum_into(c, nbins, E, nshells, bins);
    (void)hipFree(bins);
    return rc;
}

int mhit_energy_spectrum_noalloc(mhit_ctx* c, int32_t nbins, double* E, int32_t* nshells) {
    int rc;
    if ((rc = spectrum_check(c, nbins, E))) return rc;
    const int used = shells_used(c->n);
    const int nb = nbins < used ? nbins : used;
    if (nb > kScratchBins) {
        set_error("mhit_energy_spectrum_noalloc: " + std::to_string(nb) + " shells exceed the " +
                  std::to_string(kScratchBins) + "-shell scratch (ask for fewer bins)");
        return MHIT_ERR_ARG;
    }
    double* bins = nullptr;
    if ((rc = scratch_on(c->device, &bins))) return rc;
    return spectrum_into(c, nbins, E, nshells, bins);
}

}  // extern "C"
