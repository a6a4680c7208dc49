// stencil.hip -- finite-difference passes of the MHIT36 timestep (gfx950).
//
// Each kernel restates the reference loop it cites (aroccon/MHIT36_mixedp,
// multi/main.f90) with the reference's operand order; the library is built
// without FP contraction.  Halo exchanges are replaced by periodic index
// wrap.  The velocity state is stored with a deferred mean: the reference
// removes the mean from u,v,w after the correction (main.f90:977-981); here
// the correction writes u + mean and every reader subtracts mean on load,
// which yields the same FP64 values without a second pass over u,v,w.
#include "internal.hpp"

#include <algorithm>
#include <cmath>
#include <vector>

namespace mhit {

#define MHIT_CELL_INDEX(g)                                   \
    const int n = (g).n;                                     \
    const int i = blockIdx.x * 64 + threadIdx.x;             \
    const int j = blockIdx.y * 4 + threadIdx.y;              \
    const int k = blockIdx.z;                                \
    if (i >= n || j >= n) return;                            \
    const int ip = wrap_p(i, n), im = wrap_m(i, n);          \
    const int jp = wrap_p(j, n), jm = wrap_m(j, n);          \
    const int kp = wrap_p(k, n), km = wrap_m(k, n);          \
    (void)ip; (void)im; (void)jp; (void)jm; (void)kp; (void)km; \
    const size_t q = idx3(i, j, k, n)

// ----------------------------------------------------------------- ACDI
// P1, main.f90:522-534 (all points)
__global__ __launch_bounds__(256)
void k_acdi_psi(const double* __restrict__ phi, double* __restrict__ psi,
                double* __restrict__ tpsi, Grid g, const DevScalars* __restrict__ S) {
    if (S->halted) return;
    MHIT_CELL_INDEX(g);
    const double val = fmin(phi[q], 1.0);
    const double ps = g.eps * log((val + g.enm) / (1.0 - val + g.enm));
    psi[q] = ps;
    tpsi[q] = tanh(0.5 * ps * g.epsi);
}

// P2, main.f90:536-564: convective + diffusive flux, raw normals
__global__ __launch_bounds__(256)
void k_acdi_rhs(const double* __restrict__ u, const double* __restrict__ v,
                const double* __restrict__ w, const double* __restrict__ phi,
                const double* __restrict__ psi, double* __restrict__ rphi,
                double* __restrict__ nx, double* __restrict__ ny, double* __restrict__ nz,
                Grid g, const DevScalars* __restrict__ S) {
    if (S->halted) return;
    MHIT_CELL_INDEX(g);
    const double m0 = S->mean[0], m1 = S->mean[1], m2 = S->mean[2];
    const double gamma = 1.0 * S->gumax;
    const double dxi = g.dxi, ddxi = g.ddxi, eps = g.eps;
    const double uc = u[q] - m0, up = u[idx3(ip, j, k, n)] - m0;
    const double vc = v[q] - m1, vp = v[idx3(i, jp, k, n)] - m1;
    const double wc = w[q] - m2, wp = w[idx3(i, j, kp, n)] - m2;
    const double pc = phi[q];
    const double pxp = phi[idx3(ip, j, k, n)], pxm = phi[idx3(im, j, k, n)];
    const double pyp = phi[idx3(i, jp, k, n)], pym = phi[idx3(i, jm, k, n)];
    const double pzp = phi[idx3(i, j, kp, n)], pzm = phi[idx3(i, j, km, n)];
    double r = -(up * 0.5 * (pxp + pc) - uc * 0.5 * (pc + pxm)) * dxi
               - (vp * 0.5 * (pyp + pc) - vc * 0.5 * (pc + pym)) * dxi
               - (wp * 0.5 * (pzp + pc) - wc * 0.5 * (pc + pzm)) * dxi
               + gamma * (eps * (pxp - 2.0 * pc + pxm) * ddxi +
                          eps * (pyp - 2.0 * pc + pym) * ddxi +
                          eps * (pzp - 2.0 * pc + pzm) * ddxi);
    rphi[q] = r;
    nx[q] = (psi[idx3(ip, j, k, n)] - psi[idx3(im, j, k, n)]);
    ny[q] = (psi[idx3(i, jp, k, n)] - psi[idx3(i, jm, k, n)]);
    nz[q] = (psi[idx3(i, j, kp, n)] - psi[idx3(i, j, km, n)]);
}

// P3, main.f90:582-593
__global__ __launch_bounds__(256)
void k_acdi_normalize(double* __restrict__ nx, double* __restrict__ ny, double* __restrict__ nz,
                      Grid g, const DevScalars* __restrict__ S) {
    if (S->halted) return;
    MHIT_CELL_INDEX(g);
    const double a = nx[q], b = ny[q], c = nz[q];
    const double normag = 1.0 / (sqrt(a * a + b * b + c * c) + g.enm);
    nx[q] = a * normag;
    ny[q] = b * normag;
    nz[q] = c * normag;
}

// P4 + P5, main.f90:596-630: sharpening flux and AB2 of phi (in place)
__global__ __launch_bounds__(256)
void k_acdi_update(double* __restrict__ phi, const double* __restrict__ rphi_in,
                   double* __restrict__ rphi_o, const double* __restrict__ T,
                   const double* __restrict__ nx, const double* __restrict__ ny,
                   const double* __restrict__ nz, Grid g, const DevScalars* __restrict__ S) {
    if (S->halted) return;
    MHIT_CELL_INDEX(g);
    const double gamma = 1.0 * S->gumax;
    const double alpha = S->alpha, beta = S->beta, dxi = g.dxi;
    const double Txp = T[idx3(ip, j, k, n)], Txm = T[idx3(im, j, k, n)];
    const double Typ = T[idx3(i, jp, k, n)], Tym = T[idx3(i, jm, k, n)];
    const double Tzp = T[idx3(i, j, kp, n)], Tzm = T[idx3(i, j, km, n)];
    double r = rphi_in[q] -
               gamma * ((0.25 * (1.0 - Txp * Txp) * nx[idx3(ip, j, k, n)] -
                         0.25 * (1.0 - Txm * Txm) * nx[idx3(im, j, k, n)]) * 0.5 * dxi +
                        (0.25 * (1.0 - Typ * Typ) * ny[idx3(i, jp, k, n)] -
                         0.25 * (1.0 - Tym * Tym) * ny[idx3(i, jm, k, n)]) * 0.5 * dxi +
                        (0.25 * (1.0 - Tzp * Tzp) * nz[idx3(i, j, kp, n)] -
                         0.25 * (1.0 - Tzm * Tzm) * nz[idx3(i, j, km, n)]) * 0.5 * dxi);
    phi[q] = phi[q] + g.dt * (alpha * r - beta * rphi_o[q]);
    rphi_o[q] = r;
}

int launch_acdi(mhit_ctx* c) {
    CellLaunch L(c->n);
    k_acdi_psi<<<L.grid, L.block, 0, c->stream>>>(c->phi, c->psi, c->tanh_psi, c->g, c->S);
    prof_mark(c, ST_ACDI_PSI);
    k_acdi_rhs<<<L.grid, L.block, 0, c->stream>>>(c->u, c->v, c->w, c->phi, c->psi, c->rhsphi,
                                                  c->normx, c->normy, c->normz, c->g, c->S);
    prof_mark(c, ST_ACDI_RHS);
    k_acdi_normalize<<<L.grid, L.block, 0, c->stream>>>(c->normx, c->normy, c->normz, c->g, c->S);
    prof_mark(c, ST_ACDI_NORM);
    k_acdi_update<<<L.grid, L.block, 0, c->stream>>>(c->phi, c->rhsphi, c->rhsphi_o, c->tanh_psi,
                                                     c->normx, c->normy, c->normz, c->g, c->S);
    prof_mark(c, ST_ACDI_UPDATE);
    MHIT_HIP_TRY(hipGetLastError());
    return MHIT_OK;
}

// ------------------------------------------------------------------ CSF
// S1, main.f90:721-743 (phi already advanced)
__global__ __launch_bounds__(256)
void k_csf(const double* __restrict__ phi, double* __restrict__ fx, double* __restrict__ fy,
           double* __restrict__ fz, Grid g, const DevScalars* __restrict__ S) {
    if (S->halted) return;
    MHIT_CELL_INDEX(g);
    const double ph = phi[q];
    const double pxp = phi[idx3(ip, j, k, n)], pxm = phi[idx3(im, j, k, n)];
    const double pyp = phi[idx3(i, jp, k, n)], pym = phi[idx3(i, jm, k, n)];
    const double pzp = phi[idx3(i, j, kp, n)], pzm = phi[idx3(i, j, km, n)];
    const double chempot = ph * (1.0 - ph) * (1.0 - 2.0 * ph) * g.epsi -
                           g.eps * (pxp + pxm + pyp + pym + pzp + pzm - 6.0 * ph) * g.ddxi;
    fx[q] = 6.0 * g.sigma * chempot * 0.5 * (pxp - pxm) * g.dxi;
    fy[q] = 6.0 * g.sigma * chempot * 0.5 * (pyp - pym) * g.dxi;
    fz[q] = 6.0 * g.sigma * chempot * 0.5 * (pzp - pzm) * g.dxi;
}

// ------------------------------------------------------------------- NS
// N1 (main.f90:658-717) fused with the face force + AB2 of S2
// (main.f90:760-780) or with N2 (783-796).  Writes u* to us,vs,ws.
template <bool PHI>
__global__ __launch_bounds__(256)
void k_ns(const double* __restrict__ u, const double* __restrict__ v, const double* __restrict__ w,
          const double* __restrict__ fx, const double* __restrict__ fy, const double* __restrict__ fz,
          double* __restrict__ ru_o, double* __restrict__ rv_o, double* __restrict__ rw_o,
          double* __restrict__ us, double* __restrict__ vs, double* __restrict__ ws,
          const double* __restrict__ mysin, const double* __restrict__ mycos,
          Grid g, const DevScalars* __restrict__ S) {
    if (S->halted) return;
    MHIT_CELL_INDEX(g);
    const double m0 = S->mean[0], m1 = S->mean[1], m2 = S->mean[2];
    const double alpha = S->alpha, beta = S->beta;
    const double dxi = g.dxi, ddxi = g.ddxi, mu = g.mu, rhoi = g.rhoi;
#define U(a, b, c) (u[idx3(a, b, c, n)] - m0)
#define V(a, b, c) (v[idx3(a, b, c, n)] - m1)
#define W(a, b, c) (w[idx3(a, b, c, n)] - m2)
    const double u0 = U(i, j, k), v0 = V(i, j, k), w0 = W(i, j, k);
    const double uxp = U(ip, j, k), uxm = U(im, j, k), uyp = U(i, jp, k), uym = U(i, jm, k);
    const double uzp = U(i, j, kp), uzm = U(i, j, km);
    const double vxp = V(ip, j, k), vxm = V(im, j, k), vyp = V(i, jp, k), vym = V(i, jm, k);
    const double vzp = V(i, j, kp), vzm = V(i, j, km);
    const double wxp = W(ip, j, k), wxm = W(im, j, k), wyp = W(i, jp, k), wym = W(i, jm, k);
    const double wzp = W(i, j, kp), wzm = W(i, j, km);
    double h11 = (uxp + u0) * (uxp + u0) - (u0 + uxm) * (u0 + uxm);
    double h12 = (uyp + u0) * (vyp + V(im, jp, k)) - (u0 + uym) * (v0 + vxm);
    double h13 = (uzp + u0) * (wzp + W(im, j, kp)) - (u0 + uzm) * (w0 + wxm);
    double h21 = (uxp + U(ip, jm, k)) * (vxp + v0) - (u0 + uym) * (v0 + vxm);
    double h22 = (vyp + v0) * (vyp + v0) - (v0 + vym) * (v0 + vym);
    double h23 = (wzp + W(i, jm, kp)) * (vzp + v0) - (w0 + wym) * (v0 + vzm);
    double h31 = (wxp + w0) * (uxp + U(ip, j, km)) - (w0 + wxm) * (u0 + uzm);
    double h32 = (vyp + V(i, jp, km)) * (wyp + w0) - (v0 + vzm) * (w0 + wym);
    double h33 = (wzp + w0) * (wzp + w0) - (w0 + wzm) * (w0 + wzm);
#undef U
#undef V
#undef W
    h11 = h11 * 0.25 * dxi; h12 = h12 * 0.25 * dxi; h13 = h13 * 0.25 * dxi;
    h21 = h21 * 0.25 * dxi; h22 = h22 * 0.25 * dxi; h23 = h23 * 0.25 * dxi;
    h31 = h31 * 0.25 * dxi; h32 = h32 * 0.25 * dxi; h33 = h33 * 0.25 * dxi;
    double ru = -(h11 + h12 + h13);
    double rv = -(h21 + h22 + h23);
    double rw = -(h31 + h32 + h33);
    h11 = mu * (uxp - 2.0 * u0 + uxm) * ddxi;
    h12 = mu * (uyp - 2.0 * u0 + uym) * ddxi;
    h13 = mu * (uzp - 2.0 * u0 + uzm) * ddxi;
    h21 = mu * (vxp - 2.0 * v0 + vxm) * ddxi;
    h22 = mu * (vyp - 2.0 * v0 + vym) * ddxi;
    h23 = mu * (vzp - 2.0 * v0 + vzm) * ddxi;
    h31 = mu * (wxp - 2.0 * w0 + wxm) * ddxi;
    h32 = mu * (wyp - 2.0 * w0 + wym) * ddxi;
    h33 = mu * (wzp - 2.0 * w0 + wzm) * ddxi;
    ru = ru + (h11 + h12 + h13) * rhoi;
    rv = rv + (h21 + h22 + h23) * rhoi;
    rw = rw + (h31 + h32 + h33) * rhoi;
    // ABC forcing: kg = k+2, jg = j+2 in Fortran indexing -> table k+1, j+1
    ru = ru + g.f3 * mysin[k + 1] + g.f2 * mycos[j + 1];
    rv = rv + g.f1 * mysin[i] + g.f3 * mycos[k + 1];
    rw = rw + g.f2 * mysin[j + 1] + g.f1 * mycos[i];
    if (PHI) {
        ru = ru + 0.5 * (fx[idx3(im, j, k, n)] + fx[q]) * rhoi;
        rv = rv + 0.5 * (fy[idx3(i, jm, k, n)] + fy[q]) * rhoi;
        rw = rw + 0.5 * (fz[idx3(i, j, km, n)] + fz[q]) * rhoi;
    }
    const double dt = g.dt;
    us[q] = u0 + dt * (alpha * ru - beta * ru_o[q]);
    vs[q] = v0 + dt * (alpha * rv - beta * rv_o[q]);
    ws[q] = w0 + dt * (alpha * rw - beta * rw_o[q]);
    ru_o[q] = ru;
    rv_o[q] = rv;
    rw_o[q] = rw;
}

int launch_ns(mhit_ctx* c) {
    CellLaunch L(c->n);
    if (c->P.phiflag) {
        k_csf<<<L.grid, L.block, 0, c->stream>>>(c->phi, c->fxst, c->fyst, c->fzst, c->g, c->S);
        prof_mark(c, ST_CSF);
        k_ns<true><<<L.grid, L.block, 0, c->stream>>>(
            c->u, c->v, c->w, c->fxst, c->fyst, c->fzst, c->rhsu_o, c->rhsv_o, c->rhsw_o,
            c->us, c->vs, c->ws, c->mysin, c->mycos, c->g, c->S);
    } else {
        k_ns<false><<<L.grid, L.block, 0, c->stream>>>(
            c->u, c->v, c->w, nullptr, nullptr, nullptr, c->rhsu_o, c->rhsv_o, c->rhsw_o,
            c->us, c->vs, c->ws, c->mysin, c->mycos, c->g, c->S);
    }
    prof_mark(c, ST_NS);
    MHIT_HIP_TRY(hipGetLastError());
    return MHIT_OK;
}

// ----------------------------------------------------------- correction
// C, main.f90:942-962: u = u* - dt/rho (p - p(-1)) dxi with the pressure
// promoted to FP64, plus per-block sums and maxima of the corrected u,v,w.
// Bound by HBM: 52 (FP32 p) or 56 bytes per cell.
//
// Summation order.  The mean enters every velocity of the next step.  With
// the FP32 Poisson a last-bit change of it flips roundings of div u* and so
// replaces the whole FP32 rounding noise of p by another sample (2.5e-7 of
// p, 1e-9 of u after ten steps at 256^3).  Its order is therefore fixed by
// the grid size alone: 64 x 8 tiles (32 x 16 where n is a multiple of 32 but
// not of 64: 96^3), chunks of correct_zc planes summed from the bottom up,
// partials by 1024 interleaved runs.  With the FP64 Poisson the order is
// fixed by the grid size too, but free to follow the faster sweep.
//
// k_correct takes a few planes of loads in flight per thread and p's
// neighbours through the caches, without LDS and barriers.  (Marching one
// plane at a time with p in LDS behind a barrier, in a running step: 64^3
// 8.6 -> 7.0 us, 128^3 FP32 38 -> 24 us, 192^3 FP64 102 -> 70 us.)  From
// 256^3 its workgroups are wide and flat, so that the dispatch order sweeps
// memory front to back.  FP64: 128 x 4 columns of two planes, 512^3 1.36 ->
// 1.18 ms (6.3 TB/s).  FP32: rows of 256 cells (128 x 2 where n is no
// multiple of 256) over the order's chunk, 512^3 1.27 -> 1.20 ms, 384^3 0.59
// -> 0.54, 256^3 0.172 -> 0.158 (5.5 TB/s) against the march; a wave writes
// its row's sums and k_fin_rows (5 us at 256^3 and 384^3, 11 at 512^3) adds
// them up as an 8-row tile would.
// The rows start where a launch covers as many cells as 256^3, so that an
// ensemble's batches of 128^3 take them too (eight planes in flight: 16 x
// 64^3 + 16 x 96^3 + 16 x 128^3 2.44 -> 2.36 ms per step, 16 x 128^3 1.51 ->
// 1.48; 128^3 alone 0.109 -> 0.113, so not there).
constexpr int CO_NT = 512;                    // threads per workgroup of the 8-row tile
struct CorrShape { int mx, my, zc; bool rows; };
static CorrShape correct_shape(int n, bool fp32, int nb) {
    if (!fp32 && n >= 64) return {n >= 256 ? 128 : (n % 64 == 0 ? 64 : 32), n % 64 == 0 ? 4 : 16,
                                  n >= 256 ? 2 : 4, false};
    const int mx = (n > 64 && n % 64 != 0 && n % 32 == 0) ? 32 : 64, my = CO_NT / mx;
    // the longest of 32, 16, ... 2 planes with at least 256 workgroups
    const long long tiles = (long long)div_up(n, mx) * div_up(n, my);
    int zc = n >= 512 ? 16 : 32;
    while (n < 512 && zc > 2 && tiles * div_up(n, zc) < 256) zc /= 2;
    if (n % 128 == 0 && (long long)n * n * n * nb >= 256LL * 256 * 256)
        return {n % 256 == 0 ? 256 : 128, n % 256 == 0 ? 1 : 2, zc, true};
    return {mx, my, zc < n ? zc : n, false};
}

static dim3 correct_grid(int n, bool fp32, int nb) {
    const CorrShape s = correct_shape(n, fp32, nb);
    return dim3(div_up(n, s.mx), div_up(n, s.my), div_up(n, s.zc));
}

// Arguments of one box (a batched launch reads a table of them).
template <typename T>
struct CorrArgs {
    const double *us, *vs, *ws;
    const T* p;
    double *u, *v, *w, *partials;
    Grid g;
    const DevScalars* S;
    int zc, xcd;
};

template <typename T, int MX, int MY, int U, bool ROWS = false>
__global__ __launch_bounds__(MX * MY)
void k_correct(CorrArgs<T> one, const CorrArgs<T>* __restrict__ tab, int nbox) {
    const Blk blk = launch_blk(nbox);
    CorrArgs<T> A = one;
    if (tab) A = tab[blk.box];
    const MHIT_GLOBAL double* __restrict__ us = gmem(A.us);
    const MHIT_GLOBAL double* __restrict__ vs = gmem(A.vs);
    const MHIT_GLOBAL double* __restrict__ ws = gmem(A.ws);
    const MHIT_GLOBAL T* __restrict__ p = gmem(A.p);
    MHIT_GLOBAL double* __restrict__ u = gmem(A.u);
    MHIT_GLOBAL double* __restrict__ v = gmem(A.v);
    MHIT_GLOBAL double* __restrict__ w = gmem(A.w);
    MHIT_GLOBAL double* __restrict__ partials = gmem(A.partials);
    const Grid g = A.g;
    const MHIT_GLOBAL DevScalars* __restrict__ S = gmem(A.S);
    constexpr int NT = MX * MY;          // U planes in flight
    __shared__ double red[6][NT / 64];
    const int n = g.n;
    const int tid = threadIdx.y * MX + threadIdx.x;
    int tbx, tby, tbz;
    xcd_tile(tbx, tby, tbz, blk, A.xcd);
    const int i = tbx * MX + threadIdx.x, j = tby * MY + threadIdx.y;
    const int z0 = tbz * A.zc, z1 = min(z0 + A.zc, n);
    if (S->halted) return;               // the finalize pass reads no partials then
    const double dtr = g.dt / g.rho;
    double su = 0.0, sv = 0.0, sw = 0.0;
    double mu_ = -INFINITY, mv_ = -INFINITY, mw_ = -INFINITY;
    if (i < n && j < n) {
        // in-plane offsets of the cell and of its -x and -y neighbours
        const int o = j * n + i, ox = j * n + wrap_m(i, n), oy = wrap_m(j, n) * n + i;
        const size_t plane = (size_t)n * n;
        T pm = p[wrap_m(z0, n) * plane + o];
        for (int k = z0; k < z1; k += U) {
            T pc[U], px[U], py[U];
            double uq[U], vq[U], wq[U];
#pragma unroll
            for (int t = 0; t < U; t++) {
                if (k + t >= z1) continue;
                const size_t b = (k + t) * plane;
                pc[t] = p[b + o]; px[t] = p[b + ox]; py[t] = p[b + oy];
                uq[t] = ld_once(&us[b + o]); vq[t] = ld_once(&vs[b + o]); wq[t] = ld_once(&ws[b + o]);
            }
#pragma unroll
            for (int t = 0; t < U; t++) {
                if (k + t >= z1) continue;
                const size_t q = (k + t) * plane + o;
                const double c = (double)pc[t];
                const double uu = uq[t] - dtr * (c - (double)px[t]) * g.dxi;
                const double vv = vq[t] - dtr * (c - (double)py[t]) * g.dxi;
                const double ww = wq[t] - dtr * (c - (double)pm) * g.dxi;
                st_once(&u[q], uu); st_once(&v[q], vv); st_once(&w[q], ww);
                su += uu; sv += vv; sw += ww;
                mu_ = fmax(mu_, uu); mv_ = fmax(mv_, vv); mw_ = fmax(mw_, ww);
                pm = pc[t];
            }
        }
    }
    su = wave_sum(su); sv = wave_sum(sv); sw = wave_sum(sw);
    mu_ = wave_max(mu_); mv_ = wave_max(mv_); mw_ = wave_max(mw_);
    if constexpr (ROWS) {
        // [chunk][row][64-cell segment]; the waves hold one segment each
        if ((tid & 63) == 0) {
            const double r[6] = {su, sv, sw, mu_, mv_, mw_};
            const size_t b = ((size_t)tbz * n + j) * (n / 64) + i / 64;
            for (int f = 0; f < 6; f++) partials[b * 6 + f] = r[f];
        }
        return;
    }
    const int wv = tid >> 6;
    if ((tid & 63) == 0) {
        red[0][wv] = su; red[1][wv] = sv; red[2][wv] = sw;
        red[3][wv] = mu_; red[4][wv] = mv_; red[5][wv] = mw_;
    }
    __syncthreads();
    if (tid < 6) {
        const int f = tid;
        double r = red[f][0];
        for (int t = 1; t < NT / 64; t++) r = (f < 3) ? r + red[f][t] : fmax(r, red[f][t]);
        // partials in tile order, so the reduction order does not depend on
        // the workgroup order (xcd_tile)
        const size_t b = ((size_t)tbz * blk.ny + tby) * blk.nx + tbx;
        partials[b * 6 + f] = r;
    }
}

template <typename T>
static CorrArgs<T> corr_args(mhit_ctx* c) {
    CorrArgs<T> a;
    a.us = c->us; a.vs = c->vs; a.ws = c->ws;
    a.p = (const T*)c->pres;
    a.u = c->u; a.v = c->v; a.w = c->w;
    a.partials = c->partials;
    a.g = c->g;
    a.S = c->S;
    a.zc = correct_shape(c->n, c->fp32, 1).zc;   // the same for any nb
    // XCD tile order for small boxes (96^3 10.9 against 11.3 us, 512^3 FP32
    // 1.24 against 1.17 ms); the partials are indexed by tile, so the order
    // changes no bit
    a.xcd = c->n < 192;
    return a;
}

template <typename T>
static void go_correct(int n, const CorrArgs<T>& one, const CorrArgs<T>* tab, int nb, hipStream_t st) {
    constexpr bool F32 = sizeof(T) == 4;
    const CorrShape sh = correct_shape(n, F32, nb);
    dim3 grid = correct_grid(n, F32, nb);
    grid.z *= nb;
    const dim3 block(sh.mx, sh.my, 1);
    if constexpr (F32) {
        if (sh.rows) {
            if (n == 128) k_correct<T, 128, 2, 8, true><<<grid, block, 0, st>>>(one, tab, nb);
            else if (sh.mx == 128) k_correct<T, 128, 2, 2, true><<<grid, block, 0, st>>>(one, tab, nb);
            else if (n >= 512) k_correct<T, 256, 1, 2, true><<<grid, block, 0, st>>>(one, tab, nb);
            else k_correct<T, 256, 1, 8, true><<<grid, block, 0, st>>>(one, tab, nb);
            return;
        }
    } else {
        if (sh.mx == 128) {
            k_correct<T, 128, 4, 2><<<grid, block, 0, st>>>(one, tab, nb);
            return;
        }
        if (sh.my == 4) {
            k_correct<T, 64, 4, 2><<<grid, block, 0, st>>>(one, tab, nb);
            return;
        }
    }
    if (sh.mx == 32) k_correct<T, 32, 16, 2><<<grid, block, 0, st>>>(one, tab, nb);
    else if (n >= 192) k_correct<T, 64, 8, 4><<<grid, block, 0, st>>>(one, tab, nb);
    else k_correct<T, 64, 8, 2><<<grid, block, 0, st>>>(one, tab, nb);
}

int launch_correct(mhit_ctx* c) {
    if (c->fp32) go_correct<float>(c->n, corr_args<float>(c), nullptr, 1, c->stream);
    else go_correct<double>(c->n, corr_args<double>(c), nullptr, 1, c->stream);
    prof_mark(c, ST_CORRECT);
    MHIT_HIP_TRY(hipGetLastError());
    return MHIT_OK;
}

template <typename T>
static int correct_batch(mhit_ctx* const* boxes, int nb, ArgArena& arena, hipStream_t st) {
    std::vector<CorrArgs<T>> t(nb);
    for (int b = 0; b < nb; b++) t[b] = corr_args<T>(boxes[b]);
    const CorrArgs<T>* tab = arena.put(t.data(), nb);
    if (!tab) { set_error("batched launch: argument arena full"); return MHIT_ERR_STATE; }
    go_correct<T>(boxes[0]->n, t[0], tab, nb, st);
    MHIT_HIP_TRY(hipGetLastError());
    return MHIT_OK;
}

int launch_correct_batch(mhit_ctx* const* boxes, int nb, ArgArena& arena, hipStream_t st) {
    mhit_ctx* c = boxes[0];
    for (int b = 1; b < nb; b++)
        if (boxes[b]->n != c->n || boxes[b]->fp32 != c->fp32) {
            set_error("batched correction: boxes differ in size or precision");
            return MHIT_ERR_ARG;
        }
    return c->fp32 ? correct_batch<float>(boxes, nb, arena, st) : correct_batch<double>(boxes, nb, arena, st);
}

// Finalize: means (main.f90:964-974), signed max after the mean removal
// (998-1002, max(u - m) = max(u) - m as rounding is monotone), CFL
// (1003-1006), AB2 switch (801-802).  One workgroup, fixed reduction order:
// thread t adds up partials t, t + 1024, ..., then a tree over the threads.
// k_fin_rows first makes those 1024 sums from row sums (the FP32 sweeps of
// large boxes), and above kFinMost partials (the FP64 ones) k_fin_parts
// first adds up runs of kFinPart: one workgroup alone takes 16 us for the
// 16,384 partials of 512^3.
constexpr int kFinMost = 4096, kFinPart = 64, kFinRuns = 1024;

// partials of the correction's workgroups (waves, for row sums)
int correct_block_count(int n, bool fp32, int nb) {
    const CorrShape s = correct_shape(n, fp32, nb);
    if (s.rows) return (n / 64) * n * div_up(n, s.zc);
    const dim3 g = correct_grid(n, fp32, nb);
    return (int)(g.x * g.y * g.z);
}
// sums that k_finalize starts from instead of the partials (0: none)
static int fin_parts(int n, bool fp32, int nb) {
    const int parts = correct_block_count(n, fp32, nb);
    if (correct_shape(n, fp32, nb).rows) return std::min(kFinRuns, parts / 8);
    return parts > kFinMost ? div_up(parts, kFinPart) : 0;
}
// space for the partials, in doubles: the correction's, then their sums, of
// a box alone or in a launch of any number of boxes
size_t correct_partials(int n, bool fp32) {
    auto need = [&](int nb) { return (size_t)(correct_block_count(n, fp32, nb) + fin_parts(n, fp32, nb)) * 6; };
    return std::max(need(1), need(1 << 20));
}

struct FinArgs {
    double* partials;
    int nblocks, nparts, cfl_abort;   // partials, and sums of runs of them (0: none)
    Grid g;
    DevScalars* S;
};

// A wave per run of kFinPart partials; blockIdx.y is the box of a batched
// launch.
__global__ __launch_bounds__(256)
void k_fin_parts(FinArgs one, const FinArgs* __restrict__ tab) {
    FinArgs A = one;
    if (tab) A = tab[blockIdx.y];
    if (gmem(A.S)->halted) return;
    const int run = blockIdx.x * 4 + (threadIdx.x >> 6), b = run * kFinPart + (threadIdx.x & 63);
    if (run >= A.nparts) return;
    MHIT_GLOBAL double* partials = gmem(A.partials);
    const bool on = b < A.nblocks;
    for (int f = 0; f < 6; f++) {
        const double x = on ? partials[(size_t)b * 6 + f] : (f < 3 ? 0.0 : -INFINITY);
        const double r = f < 3 ? wave_sum(x) : wave_max(x);
        if ((threadIdx.x & 63) == 0) partials[(size_t)(A.nblocks + run) * 6 + f] = r;
    }
}

// The row sums to the sums of the kFinRuns interleaved runs of 8-row tiles:
// tile b is segment b % (n/64) of rows 8 b' ... 8 b' + 7, b' = b / (n/64)
// (chunk by chunk), its rows are added up first to last, and run t holds
// tiles t, t + kFinRuns, ...  A thread per run and component.
__global__ __launch_bounds__(256)
void k_fin_rows(FinArgs one, const FinArgs* __restrict__ tab) {
    FinArgs A = one;
    if (tab) A = tab[blockIdx.y];
    const int q = blockIdx.x * 256 + threadIdx.x, t = q / 6, f = q - 6 * t;
    if (t >= A.nparts || gmem(A.S)->halted) return;
    MHIT_GLOBAL double* partials = gmem(A.partials);
    const int nx = A.g.n / 64, tiles = A.nblocks / 8;
    double r = f < 3 ? 0.0 : -INFINITY;
#pragma unroll 2
    for (int b = t; b < tiles; b += kFinRuns) {
        const MHIT_GLOBAL double* row = partials + ((size_t)(b / nx) * 8 * nx + b % nx) * 6 + f;
        double x[8];
#pragma unroll
        for (int j = 0; j < 8; j++) x[j] = row[(size_t)j * nx * 6];
#pragma unroll
        for (int j = 1; j < 8; j++) x[0] = f < 3 ? x[0] + x[j] : fmax(x[0], x[j]);
        r = f < 3 ? r + x[0] : fmax(r, x[0]);
    }
    partials[(size_t)(A.nblocks + t) * 6 + f] = r;
}

// One workgroup per box (blockIdx.x is the box of a batched launch).
__global__ __launch_bounds__(1024)
void k_finalize(FinArgs one, const FinArgs* __restrict__ tab) {
    FinArgs A = one;
    if (tab) A = tab[blockIdx.x];
    const Grid g = A.g;
    MHIT_GLOBAL DevScalars* __restrict__ S = gmem(A.S);
    const MHIT_GLOBAL double* __restrict__ partials = gmem(A.partials) + (A.nparts ? (size_t)A.nblocks * 6 : 0);
    const int nblocks = A.nparts ? A.nparts : A.nblocks;
    __shared__ double red[6][512];
    const int t = threadIdx.x;
    if (S->halted) {
        if (t == 0) S->skipped += 1;   // a step whose passes all returned at once
        return;
    }
    double a[6] = {0.0, 0.0, 0.0, -INFINITY, -INFINITY, -INFINITY};
    for (int b = t; b < nblocks; b += 1024) {
        for (int f = 0; f < 3; f++) a[f] += partials[(size_t)b * 6 + f];
        for (int f = 3; f < 6; f++) a[f] = fmax(a[f], partials[(size_t)b * 6 + f]);
    }
    // thread t takes up t + 512, t + 256, ..., t + 1: the first four through
    // LDS, the rest within the wave
    for (int s = 512; s >= 64; s >>= 1) {
        if (t >= s && t < 2 * s)
            for (int f = 0; f < 6; f++) red[f][t - s] = a[f];
        __syncthreads();
        if (t < s)
            for (int f = 0; f < 6; f++) a[f] = f < 3 ? a[f] + red[f][t] : fmax(a[f], red[f][t]);
        __syncthreads();
    }
    if (t >= 64) return;
    for (int s = 32; s > 0; s >>= 1)
        for (int f = 0; f < 6; f++) {
            const double x = __shfl_down(a[f], s, 64);
            a[f] = f < 3 ? a[f] + x : fmax(a[f], x);
        }
    if (t == 0) {
        const double nn = (double)g.n;
        double m[3], mx[3];
        for (int f = 0; f < 3; f++) {
            m[f] = a[f] / nn / nn / nn;
            mx[f] = a[f + 3] - m[f];
        }
        const double umax = fmax(mx[2], fmax(mx[0], mx[1]));
        S->mean[0] = m[0]; S->mean[1] = m[1]; S->mean[2] = m[2];
        S->gumax = umax;
        S->cou = umax * g.dt * g.dxi;
        S->alpha = 1.5;
        S->beta = 0.5;
        S->step += 1;
        if (A.cfl_abort && S->cou > 7.0) S->halted = 1;
    }
}

static FinArgs fin_args(mhit_ctx* c, int nb) {
    FinArgs a;
    a.partials = c->partials;
    a.nblocks = correct_block_count(c->n, c->fp32, nb);
    a.nparts = fin_parts(c->n, c->fp32, nb);
    a.cfl_abort = c->P.cfl_abort;
    a.g = c->g;
    a.S = c->S;
    return a;
}

static void go_finalize(mhit_ctx* c, const FinArgs& one, const FinArgs* tab, int nb, hipStream_t st) {
    if (one.nparts && correct_shape(c->n, c->fp32, nb).rows)
        k_fin_rows<<<dim3(div_up(one.nparts * 6, 256), nb), 256, 0, st>>>(one, tab);
    else if (one.nparts)
        k_fin_parts<<<dim3(div_up(one.nparts, 4), nb), 256, 0, st>>>(one, tab);
    k_finalize<<<nb, 1024, 0, st>>>(one, tab);
}

int launch_finalize(mhit_ctx* c) {
    go_finalize(c, fin_args(c, 1), nullptr, 1, c->stream);
    prof_mark(c, ST_FINALIZE);
    MHIT_HIP_TRY(hipGetLastError());
    return MHIT_OK;
}

int launch_finalize_batch(mhit_ctx* const* boxes, int nb, ArgArena& arena, hipStream_t st) {
    std::vector<FinArgs> t(nb);
    for (int b = 0; b < nb; b++) {
        t[b] = fin_args(boxes[b], nb);
        if (boxes[b]->n != boxes[0]->n || boxes[b]->fp32 != boxes[0]->fp32) {
            set_error("batched finalize: boxes differ in size or precision");
            return MHIT_ERR_ARG;
        }
    }
    const FinArgs* tab = arena.put(t.data(), nb);
    if (!tab) { set_error("batched launch: argument arena full"); return MHIT_ERR_STATE; }
    go_finalize(boxes[0], t[0], tab, nb, st);
    MHIT_HIP_TRY(hipGetLastError());
    return MHIT_OK;
}

// ---------------------------------------------------------- diagnostics
// Diagnostics: 64 x 8 columns per workgroup, chunks of 32 planes from
// 512^3, 16 from 256^3 and 4 below (each chunk reads two planes more; short
// chunks keep small boxes on all CUs).
constexpr int DI_MY = 8;
static int diag_zc(int n) { return n >= 512 ? 32 : n >= 256 ? 16 : 4; }
static dim3 diag_grid(int n) { return dim3(div_up(n, 64), div_up(n, DI_MY), div_up(n, diag_zc(n))); }
int diag_block_count(int n) {
    const dim3 g = diag_grid(n);
    return (int)(g.x * g.y * g.z);
}

// KE, dissipation 2 nu <S_ij S_ij> with central differences
// (post/compute_diss/main.f90:72-117, dx = lx/n, nu = mu/rho), max |D.u|
// with the divergence stencil of main.f90:841-843, phi mass and range.
// A thread marches its column up a chunk of planes with the column's three
// planes in registers; the x and y neighbours come from L1 and L2, so u, v,
// w and phi cross HBM about once.  (With a thread's planes n/16 apart, all
// neighbours from the caches and the partial sums added up on the host it
// took 0.265 ms at 256^3 with phi and 0.07 ms to read them back; now 0.201
// and 0.006 ms, 2.4 -> 1.4 ms a call at 512^3.  What is left is the latency
// of 19 loads per plane and column at six waves per SIMD.)
constexpr int NF = 8;
// sums; fields 2 and 6 maxima, 5 the minimum
__device__ __forceinline__ double diag_join(int f, double a, double b) {
    return (f == 2 || f == 6) ? fmax(a, b) : (f == 5 ? fmin(a, b) : a + b);
}
__device__ __forceinline__ double diag_start(int f) {
    return f == 5 ? INFINITY : (f == 6 ? -INFINITY : 0.0);
}

__global__ __launch_bounds__(64 * DI_MY)
void k_diag(const double* __restrict__ u, const double* __restrict__ v,
            const double* __restrict__ w, const double* __restrict__ phi,
            double* __restrict__ partials, Grid g, int zc, const DevScalars* __restrict__ S) {
    __shared__ double red[NF][DI_MY];
    const int n = g.n;
    const Blk blk = launch_blk(1);
    int tbx, tby, tbz;
    xcd_tile(tbx, tby, tbz, blk);   // neighbouring tiles' halo rows from the same L2
    const int i = tbx * 64 + threadIdx.x;
    const int j = tby * DI_MY + threadIdx.y;
    const int z0 = tbz * zc, z1 = min(z0 + zc, n);
    double acc[NF];
    for (int f = 0; f < NF; f++) acc[f] = diag_start(f);
    if (i < n && j < n) {
        const double m0 = S->mean[0], m1 = S->mean[1], m2 = S->mean[2];
        // in-plane offsets; the deferred mean cancels in every difference
        const int o = j * n + i, oxp = j * n + wrap_p(i, n), oxm = j * n + wrap_m(i, n);
        const int oyp = wrap_p(j, n) * n + i, oym = wrap_m(j, n) * n + i;
        const size_t plane = (size_t)n * n;
        const double h = 0.5 * g.dxi;
        const size_t km = wrap_m(z0, n) * plane, k0 = z0 * plane;
        double um = u[km + o], vm = v[km + o], wm = w[km + o];
        double uu = u[k0 + o], vv = v[k0 + o], ww = w[k0 + o];
        for (int k = z0; k < z1; k++) {
            const double *U = u + k * plane, *V = v + k * plane, *W = w + k * plane;
            const size_t kp = wrap_p(k, n) * plane;
            const double up = u[kp + o], vp = v[kp + o], wp = w[kp + o];
            const double uxp = U[oxp], vyp = V[oyp];
            const double uc = uu - m0, vc = vv - m1, wc = ww - m2;
            if (!isfinite(uc) || !isfinite(vc) || !isfinite(wc)) acc[7] += 1.0;
            acc[0] += uc * uc + vc * vc + wc * wc;
            const double dudx = (uxp - U[oxm]) * h, dudy = (U[oyp] - U[oym]) * h, dudz = (up - um) * h;
            const double dvdx = (V[oxp] - V[oxm]) * h, dvdy = (vyp - V[oym]) * h, dvdz = (vp - vm) * h;
            const double dwdx = (W[oxp] - W[oxm]) * h, dwdy = (W[oyp] - W[oym]) * h, dwdz = (wp - wm) * h;
            const double S12 = 0.5 * (dudy + dvdx), S13 = 0.5 * (dudz + dwdx), S23 = 0.5 * (dvdz + dwdy);
            acc[1] += dudx * dudx + dvdy * dvdy + dwdz * dwdz + 2.0 * (S12 * S12 + S13 * S13 + S23 * S23);
            const double dv = ((uxp - uu) + (vyp - vv) + (wp - ww)) * g.dxi;
            acc[2] = fmax(acc[2], fabs(dv));
            if (phi) {
                const double ph = phi[k * plane + o];
                if (!isfinite(ph)) acc[7] += 1.0;
                acc[3] += ph;
                acc[5] = fmin(acc[5], ph);
                acc[6] = fmax(acc[6], ph);
            }
            um = uu; vm = vv; wm = ww;
            uu = up; vv = vp; ww = wp;
        }
    }
    for (int f = 0; f < NF; f++) {
        double x = acc[f];
        for (int off = 32; off > 0; off >>= 1) x = diag_join(f, x, __shfl_xor(x, off, 64));
        acc[f] = x;
    }
    if ((threadIdx.x & 63) == 0)
        for (int f = 0; f < NF; f++) red[f][threadIdx.y] = acc[f];
    __syncthreads();
    if (threadIdx.y == 0 && threadIdx.x < NF) {
        const int f = threadIdx.x;
        double r = red[f][0];
        for (int t = 1; t < DI_MY; t++) r = diag_join(f, r, red[f][t]);
        const size_t b = ((size_t)tbz * blk.ny + tby) * blk.nx + tbx;
        partials[b * NF + f] = r;
    }
}

// The workgroups' partials to out[0, NF), a workgroup per field.
__global__ __launch_bounds__(1024)
void k_diag_sum(const double* __restrict__ partials, int nb, double* __restrict__ out) {
    __shared__ double red[16];
    const int t = threadIdx.x, f = blockIdx.x;
    double r = diag_start(f);
    for (int b = t; b < nb; b += 1024) r = diag_join(f, r, partials[(size_t)b * NF + f]);
    for (int off = 32; off > 0; off >>= 1) r = diag_join(f, r, __shfl_xor(r, off, 64));
    if ((t & 63) == 0) red[t >> 6] = r;
    __syncthreads();
    if (t == 0) {
        for (int v = 1; v < 16; v++) r = diag_join(f, r, red[v]);
        out[f] = r;
        __threadfence_system();   // out is pinned host memory
    }
}

// Streaming copy at the practical HBM rate: one 16-byte vector per thread,
// nontemporal load and store, one pass over the buffer (measured 6.1 TB/s
// against 5.7 TB/s for four plain vectors per thread).
__global__ __launch_bounds__(256)
void k_copy_probe(const double2* __restrict__ src, double2* __restrict__ dst, size_t n2) {
    typedef double d2 __attribute__((ext_vector_type(2)));
    const size_t q = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (q < n2) st_once((MHIT_GLOBAL d2*)(dst + q), ld_once((const MHIT_GLOBAL d2*)(src + q)));
}

int launch_copy_probe(mhit_ctx* c, const void* src, void* dst, size_t bytes) {
    const size_t n2 = bytes / sizeof(double2);
    k_copy_probe<<<div_up((long long)n2, 256), 256, 0, c->stream>>>((const double2*)src, (double2*)dst, n2);
    MHIT_HIP_TRY(hipGetLastError());
    return MHIT_OK;
}

// Pointwise streaming over R read and W write FP64 arrays (R, W <= 8): the
// rate a kernel with a given mix of concurrent streams can reach without
// any stencil, halo or barrier (a practical ceiling for the fused passes),
// with the nontemporal stores the passes use.
struct StreamProbe {
    const double* in[8];
    double* out[8];
};

__global__ __launch_bounds__(256)
void k_stream_probe(StreamProbe p, int R, int W, size_t n) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        double s = 0.0;
#pragma unroll
        for (int r = 0; r < 8; r++)
            if (r < R) s += p.in[r][i];
#pragma unroll
        for (int w = 0; w < 8; w++)
            if (w < W) st_once(gmem(p.out[w]) + i, s + (double)w);
    }
}

int launch_stream_probe(mhit_ctx* c, const double* const* in, int R, double* const* out, int W, size_t n) {
    StreamProbe p{};
    for (int r = 0; r < R; r++) p.in[r] = in[r];
    for (int w = 0; w < W; w++) p.out[w] = out[w];
    const int blocks = (int)std::min<size_t>(32768, (n + 255) / 256);
    k_stream_probe<<<blocks, 256, 0, c->stream>>>(p, R, W, n);
    MHIT_HIP_TRY(hipGetLastError());
    return MHIT_OK;
}

int launch_diag(mhit_ctx* c, double* out) {
    const int nb = c->ndiag_blocks;
    k_diag<<<diag_grid(c->n), dim3(64, DI_MY, 1), 0, c->stream>>>(
        c->u, c->v, c->w, c->P.phiflag ? c->phi : nullptr, c->dpartials, c->g, diag_zc(c->n), c->S);
    k_diag_sum<<<NF, 1024, 0, c->stream>>>(c->dpartials, nb, c->diag_pin);
    MHIT_HIP_TRY(hipGetLastError());
    MHIT_HIP_TRY(hipStreamSynchronize(c->stream));
    for (int f = 0; f < NF; f++) out[f] = c->diag_pin[f];
    return MHIT_OK;
}

}  // namespace mhit
