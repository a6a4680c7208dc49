// drops.hip -- drop statistics from the phase field on the GPU.
//
// The reference does this after the run, from the phi/u/v/w dumps
// (post/unionfind_periodic/main.f90: mask phi >= 0.5, 6- or 26-point
// connectivity across the periodic faces, iterated min-label propagation;
// per drop: voxel count, centre as the circular mean of the cell centres
// x(i) = (i - 1/2) dx, mean velocity, volume = count dx^3) and
// post/DropCountSize/calculate_deq.f90 (d_eq = (6 V / pi)^(1/3)).
//
// Here it runs on the live state between steps:
//   1. init:    L[q] = the first cell of q's run of masked cells within its
//               wave's 64 cells of a row; -1 where not masked
//   2. merge:   for every masked cell and each "backward" neighbour (half the
//               stencil, periodic wrap), union of the two trees with an
//               atomic min link (a root is always linked to a smaller
//               index, so every chain strictly decreases: no cycles, and the
//               final root of a component is its smallest cell index)
//   3. flatten: L[q] = root(q); cells with L[q] == q are listed
//   4. the list is sorted on the host -- the drop number is the rank of the
//               smallest cell index, the reference's ordering of its final
//               (minimum) labels -- and L[root] = -2 - rank
//   5. sums:    per drop, cell count, sum of sin/cos of the cell centres on
//               each axis and the velocity sums: a wave adds up its lanes of
//               one drop, one lane adds the result with FP64 atomics
// The label array reuses the spectrum buffer (scratch between steps); the
// tables, lists and sums of up to kKeep drops belong to the context.
// Measured at 256^3 with 64 drops of 8 cells radius, before -> now: init
// 41 -> 43 us (phi read, labels written: 4.7 TB/s), merge 115 -> 55 us (one
// link per run instead of one per cell), flatten and list 62 -> 23 us, sums
// 1030 -> 31 us.
#include "internal.hpp"

#include <algorithm>
#include <cmath>
#include <vector>

namespace mhit {
int sync_scalars_public(mhit_ctx* c);
}

using namespace mhit;

namespace {

constexpr int kStats = 10;   // count, sin x, cos x, sin y, cos y, sin z, cos z, u, v, w

__device__ __forceinline__ int load_relaxed(const int* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ int find_root(const int* L, int x) {
    int y;
    while ((y = load_relaxed(&L[x])) != x) x = y;   // strictly decreasing chain
    return x;
}

__device__ void unite(int* L, int a, int b) {
    for (;;) {
        a = find_root(L, a);
        b = find_root(L, b);
        if (a == b) return;
        if (a > b) { const int t = a; a = b; b = t; }   // link the larger root to the smaller
        const int old = atomicMin(&L[b], a);
        if (old == b) return;                           // b was still a root: linked
        b = old;                                        // b had been linked meanwhile: retry lower
    }
}

__global__ __launch_bounds__(256)
void k_cc_init(const double* __restrict__ phi, int* __restrict__ L, double thr, int n, long long n3) {
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & 63;
    const bool on = q < n3 && phi[q] >= thr;
    const unsigned long long m = __ballot(on);
    // a run starts where the cell before is not masked, or in another row or wave
    const unsigned long long starts = __ballot(on && (lane == 0 || !((m >> (lane - 1)) & 1) || q % n == 0));
    if (q >= n3) return;
    int l = -1;
    if (on) l = (int)q - lane + (63 - __clzll((long long)(starts & (~0ull >> (63 - lane)))));
    L[q] = l;
}

// neighbour offsets of the backward half of the stencil
__constant__ int c_nb[13][3] = {
    {-1, 0, 0}, {0, -1, 0}, {0, 0, -1},                                  // faces
    {-1, -1, 0}, {1, -1, 0}, {-1, 0, -1}, {1, 0, -1}, {0, -1, -1}, {0, 1, -1},  // edges
    {-1, -1, -1}, {1, -1, -1}, {-1, 1, -1}, {1, 1, -1},                  // corners
};

// The cell to the left is in q's tree already unless it is in another wave
// or across the periodic face.  With faces only (nnb = 3), the union with
// the row (plane) before is left to the cell to the left where that cell is
// masked and so is its own neighbour there: the two neighbours are adjacent.
__global__ __launch_bounds__(256)
void k_cc_merge(int* __restrict__ L, int n, int nnb) {
    const long long n3 = (long long)n * n * n;
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & 63;
    const bool on = q < n3 && load_relaxed(&L[q]) >= 0;
    const unsigned long long m = __ballot(on);
    if (!on) return;
    const int i = (int)(q % n), j = (int)((q / n) % n), k = (int)(q / ((long long)n * n));
    const bool joined = lane > 0 && i > 0 && ((m >> (lane - 1)) & 1);   // to the cell to the left
    for (int t = 0; t < nnb; t++) {
        if (t == 0 && lane > 0 && i > 0) continue;   // joined, or not masked
        int a = i + c_nb[t][0], b = j + c_nb[t][1], cz = k + c_nb[t][2];
        a = a < 0 ? a + n : (a >= n ? a - n : a);
        b = b < 0 ? b + n : (b >= n ? b - n : b);
        cz = cz < 0 ? cz + n : cz;
        const long long r = ((long long)cz * n + b) * n + a;
        if (load_relaxed(&L[r]) < 0) continue;
        if (nnb == 3 && t > 0 && joined && load_relaxed(&L[r - 1]) >= 0) continue;
        unite(L, (int)q, (int)r);
    }
}

__global__ __launch_bounds__(256)
void k_cc_flatten(int* __restrict__ L, long long n3, int* __restrict__ roots, int cap, int* __restrict__ count) {
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n3 || load_relaxed(&L[q]) < 0) return;
    const int r = find_root(L, (int)q);
    if (r != (int)q) {
        L[q] = r;
        return;
    }
    const int s = atomicAdd(count, 1);
    if (s < cap) roots[s] = r;
}

// the roots again, for more of them than the first list held
__global__ __launch_bounds__(256)
void k_cc_roots(const int* __restrict__ L, long long n3, int* __restrict__ roots, int* __restrict__ count) {
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n3 && L[q] == (int)q) roots[atomicAdd(count, 1)] = (int)q;
}

__global__ __launch_bounds__(256)
void k_cc_rank(int* __restrict__ L, const int* __restrict__ roots, int nroots) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < nroots) L[roots[t]] = -2 - t;
}

// A wave sweeps kSumRows rows of a plane, 64 cells of each, and every lane
// adds up the cells of one drop; when a lane meets another drop, and at the
// end, the lanes' sums are added up drop by drop and one lane per drop adds
// to the totals.  (With a wave per 64 cells and its atomics after each,
// 0.15 ms at 256^3 with 64 drops; the totals of one drop then serialise.)
constexpr int kSumRows = 32;

__global__ __launch_bounds__(256)
void k_cc_sums(const int* __restrict__ L, const double* __restrict__ u, const double* __restrict__ v,
               const double* __restrict__ w, const double* __restrict__ ctab,
               const DevScalars* __restrict__ S, double* __restrict__ stats, int n) {
    const int lane = threadIdx.x & 63;
    const int nx = (n + 63) / 64, ny = (n + kSumRows - 1) / kSumRows;
    const int wave = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (wave >= nx * ny * n) return;
    const int i = (wave % nx) * 64 + lane, j0 = (wave / nx) % ny * kSumRows, k = wave / (nx * ny);
    const int rows = min(kSumRows, n - j0);
    const double m0 = S->mean[0], m1 = S->mean[1], m2 = S->mean[2];
    int d = -1;                 // the lane's drop
    double x[kStats] = {};
    auto flush = [&]() {
        unsigned long long todo = __ballot(d >= 0);
        while (todo) {
            const int lead = __ffsll((long long)todo) - 1;
            const int dl = __shfl(d, lead, 64);
            const unsigned long long same = __ballot(d == dl);
            todo &= ~same;
            double* st = stats + (size_t)dl * kStats;
            if (__popcll(same) == 1) {
                if (lane == lead)
                    for (int f = 0; f < kStats; f++) atomicAdd(&st[f], x[f]);
                continue;
            }
            double t[kStats];
#pragma unroll
            for (int f = 0; f < kStats; f++) t[f] = wave_sum(d == dl ? x[f] : 0.0);
            if (lane == lead)
#pragma unroll
                for (int f = 0; f < kStats; f++) atomicAdd(&st[f], t[f]);
        }
        d = -1;
#pragma unroll
        for (int f = 0; f < kStats; f++) x[f] = 0.0;
    };
    const size_t q0 = idx3(i, j0, k, n);
    constexpr int B = 8;        // rows of labels in flight
    for (int r0 = 0; r0 < rows; r0 += B) {
        int lab[B];
#pragma unroll
        for (int r = 0; r < B; r++) lab[r] = (i < n && r0 + r < rows) ? L[q0 + (size_t)(r0 + r) * n] : -1;
#pragma unroll
        for (int r = 0; r < B; r++) {
            const bool on = lab[r] != -1;
            if (__ballot(on) == 0ull) continue;
            const int e = on ? -2 - (lab[r] >= 0 ? L[lab[r]] : lab[r]) : -1;
            if (__any(on && d >= 0 && e != d)) flush();
            if (on) {
                d = e;
                const int j = j0 + r0 + r;
                const size_t q = q0 + (size_t)(r0 + r) * n;
                // ctab: sin(x_m), cos(x_m) of the cell centres x_m = (m + 1/2) dx
                x[0] += 1.0;
                x[1] += ctab[2 * i]; x[2] += ctab[2 * i + 1];
                x[3] += ctab[2 * j]; x[4] += ctab[2 * j + 1];
                x[5] += ctab[2 * k]; x[6] += ctab[2 * k + 1];
                x[7] += u[q] - m0; x[8] += v[q] - m1; x[9] += w[q] - m2;
            }
        }
    }
    flush();
}

constexpr int kKeep = 8192;   // drops that the context's own buffers hold

}  // namespace

extern "C" {

int mhit_drop_stats(mhit_ctx* c, double threshold, int connectivity, int64_t max_drops,
                    mhit_drop* out, int64_t* ndrops) {
    if (!c || !ndrops || max_drops < 0 || (max_drops > 0 && !out) ||
        (connectivity != 6 && connectivity != 26)) {
        set_error("bad arguments (connectivity is 6 or 26)");
        return MHIT_ERR_ARG;
    }
    if (!c->P.phiflag) { set_error("no phase field (phiflag = 0)"); return MHIT_ERR_STATE; }
    int rc;
    if ((rc = sync_scalars_public(c))) return rc;
    const int n = c->n;
    const long long n3 = (long long)n * n * n;
    int* L = (int*)c->spec;   // the half spectrum holds >= n^3 ints; scratch between steps
    const int nb = (int)((n3 + 255) / 256);
    const double L2PI = 2.0 * M_PI, dx = L2PI / n;

    // the context's own buffers: cell-centre table, count + list, sums
    if (!c->drop_buf) {
        std::vector<double> tab(2 * (size_t)n);
        for (int m = 0; m < n; m++) {
            tab[2 * m] = std::sin(L2PI * ((m + 0.5) * dx) / L2PI);
            tab[2 * m + 1] = std::cos(L2PI * ((m + 0.5) * dx) / L2PI);
        }
        double* buf = nullptr;
        const size_t list = (kKeep + 2) / 2;   // count and list, in doubles
        MHIT_HIP_TRY(hipMalloc((void**)&buf, (tab.size() + list + (size_t)kKeep * kStats) * sizeof(double)));
        if (copy_on_stream(c, buf, tab.data(), tab.size() * sizeof(double), hipMemcpyHostToDevice) != hipSuccess) {
            (void)hipFree(buf);
            set_error("drop statistics: table upload failed");
            return MHIT_ERR_HIP;
        }
        c->drop_buf = buf;
    }
    const double* dtab = c->drop_buf;
    int* dcount = (int*)(c->drop_buf + 2 * (size_t)n);
    int* roots = dcount + 1;
    double* stats = c->drop_buf + 2 * (size_t)n + (kKeep + 2) / 2;
    void* more = nullptr;      // list and sums of more than kKeep drops, for this call
    auto cleanup = [&]() { if (more) (void)hipFree(more); };
#define DROPS_TRY(x) do { hipError_t e_ = (x); if (e_ != hipSuccess) { (void)hipStreamSynchronize(c->stream); \
        cleanup(); set_error(std::string("HIP: ") + hipGetErrorString(e_)); return MHIT_ERR_HIP; } } while (0)
    DROPS_TRY(hipMemsetAsync(dcount, 0, sizeof(int), c->stream));
    k_cc_init<<<nb, 256, 0, c->stream>>>(c->phi, L, threshold, n, n3);
    k_cc_merge<<<nb, 256, 0, c->stream>>>(L, n, connectivity == 6 ? 3 : 13);
    k_cc_flatten<<<nb, 256, 0, c->stream>>>(L, n3, roots, kKeep, dcount);
    DROPS_TRY(hipGetLastError());
    // the count and, with it, the first drops
    std::vector<int> hr(1 + 1024);
    DROPS_TRY(copy_on_stream(c, hr.data(), dcount, hr.size() * sizeof(int), hipMemcpyDeviceToHost));
    const int count = hr[0];
    *ndrops = count;
    if (count > 0) {
        if (count > kKeep) {
            DROPS_TRY(hipMalloc(&more, (size_t)count * (kStats * sizeof(double) + sizeof(int))));
            stats = (double*)more;
            roots = (int*)(stats + (size_t)count * kStats);
            DROPS_TRY(hipMemsetAsync(dcount, 0, sizeof(int), c->stream));
            k_cc_roots<<<nb, 256, 0, c->stream>>>(L, n3, roots, dcount);
            DROPS_TRY(hipGetLastError());
        }
        if (count > 1024) {
            hr.resize(count);
            DROPS_TRY(copy_on_stream(c, hr.data(), roots, (size_t)count * sizeof(int), hipMemcpyDeviceToHost));
        } else {
            hr.erase(hr.begin());
            hr.resize(count);
        }
        std::sort(hr.begin(), hr.end());
        std::vector<double> hs((size_t)count * kStats);
        DROPS_TRY(hipMemcpyAsync(roots, hr.data(), (size_t)count * sizeof(int), hipMemcpyHostToDevice, c->stream));
        DROPS_TRY(hipMemsetAsync(stats, 0, (size_t)count * kStats * sizeof(double), c->stream));
        k_cc_rank<<<div_up(count, 256), 256, 0, c->stream>>>(L, roots, count);
        const int sweeps = div_up(n, 64) * div_up(n, kSumRows) * n;   // a wave each
        k_cc_sums<<<div_up(sweeps, 4), 256, 0, c->stream>>>(L, c->u, c->v, c->w, dtab, c->S, stats, n);
        DROPS_TRY(hipGetLastError());
        DROPS_TRY(hipMemcpyAsync(hs.data(), stats, hs.size() * sizeof(double), hipMemcpyDeviceToHost,
                                 c->stream));
        DROPS_TRY(hipStreamSynchronize(c->stream));
        const int64_t nout = std::min<int64_t>(count, max_drops);
        for (int64_t d = 0; d < nout; d++) {
            const double* s = &hs[(size_t)d * kStats];
            auto centre = [&](double sn, double cs) {
                double x = L2PI * std::atan2(sn, cs) / L2PI;
                return x < 0.0 ? x + L2PI : x;
            };
            mhit_drop& o = out[d];
            o.cells = (int64_t)std::llround(s[0]);
            o.x = centre(s[1], s[2]);
            o.y = centre(s[3], s[4]);
            o.z = centre(s[5], s[6]);
            o.u = s[7] / s[0];
            o.v = s[8] / s[0];
            o.w = s[9] / s[0];
            o.volume = s[0] * dx * dx * dx;
            o.d_eq = std::cbrt(6.0 * o.volume / M_PI);
            o.first_cell = hr[d];
        }
    }
    cleanup();
#undef DROPS_TRY
    return MHIT_OK;
}

}  // extern "C"
