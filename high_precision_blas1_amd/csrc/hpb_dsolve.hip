// hpb_dsolve.hip -- device-resident GMRES(m) and BiCGStab(L).
//
// Same algorithms and monitor rules as the C++ solver templates (which follow
// source/numerical_algos/lin_solvers/gmres.h:376-494 and bicgstabl.h:151-274), with
// every scalar of the iteration kept in device memory, so that no step waits for
// the host:
//   * dots, norms and multi-dots write (s, c) pairs to device memory; small
//     single-thread kernels turn them into the recurrence scalars in FP64 (for
//     FP32 vectors too: the Hessenberg matrix, the Givens rotations, the back
//     substitution and BiCGStab's L x L minimal-residual solve are FP64);
//   * GMRES: one restart cycle (restart residual, m Arnoldi steps with two classical
//     Gram-Schmidt projections each, the second delayed into the next step's pass or,
//     with gram_schmidt 2, taken when the first asks for it; back substitution,
//     x += V y) is captured once as a hipGraph and replayed; the host reads one flag
//     per cycle;
//   * BiCGStab(L): one cycle (L BiCG steps, the MR part, the optional true
//     residual, the norm check) per graph; the host reads the flag every few
//     cycles;
//   * convergence, breakdown and the iteration cap raise device flags; every
//     kernel of a graph tests its flag on entry, so replays after the end do no
//     work and leave x untouched.
// MR part of BiCGStab(L): the normal equations of min ||r_0 - sum_j g_j r_j||,
// G g = c with G_ij = (r_i, r_j), c_i = (r_i, r_0) (1 <= i, j <= L), are formed by
// fused compensated multi-dots and solved by Cholesky in FP64; in exact arithmetic
// this is the reference's modified Gram-Schmidt solution (bicgstabl.h:224-245),
// and x, r_0, u_0 are then updated in one pass.
#include <hip/hip_runtime.h>

#include <chrono>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "hpb_device.hpp"
#include "hpb_internal.hpp"
#include "hpb_sdia.hpp"

namespace hpb {
namespace {

constexpr int DB = 256;        // threads per block of the vector kernels

// Threads of the one-block kernels that merge a fused kernel's partials: bound by the
// chain of merges a thread runs before the block's reduction, and below by the start of
// the block.  BiCGStab(4) of 872k rows and BiCGStab(2) of 10.5k rows, per iteration: 256
// threads 80.5 and 33.3 us, 512 threads 77.4 and 34.1, 1024 threads 77.8 and 35.9.
constexpr int FB = 512;
// Entries of a CSR matrix from which rows of more than 4 lanes are formed from staged
// tiles: below, too few tiles for the CUs.  BiCGStab(2) FP64 on uneven rows, us per
// iteration, direct / staged: 100 000 rows of 30 (3.0 M entries) 75 / 78, 300 000 of 12
// (3.7 M) 98 / 89, 378 699 of 13 117 / 106, 150 000 of 40 113 / 104; BiCGStab(4), 600 000
// of 24, 233 / 201; FP32 inner iterations, 300 000 of 20, 94 / 72.
constexpr long DS_WIDE_NNZ = 3500000;
constexpr int MAXB = 256;      // GMRES basis vectors (m + 1 <= 256)
constexpr int MAXL = 8;        // BiCGStab(L) basis in the device path

struct dstate {
    double tol, bnorm, rnorm;
    double rlast;   // reliable updates: FP64 true residual norm at the last update
    int restart;    // reliable updates: the FP32 iteration restarts from the new residual
    double rho, alpha, omega;
    int iters, max_iters, min_iters, cycles;
    int done, stop, converged, breakdown, invalid;
    int cycle_len, hist_len, hist_cap, recalc_freq, skip_recalc;
    int early_exit, basis;
    // reliable updates: the FP32 residual is the true one / rscale, and x64 gains
    // xscale * x32 (both powers of two: 1 in every other solve)
    double rscale, xscale;
    double wn2;   // GMRES selective reorthogonalisation: ||w||^2 before the projection
    int skip1;    // ... 1 when the second Gram-Schmidt pass is not needed (or the cycle stopped)
};

template <typename T>
__device__ __forceinline__ double dval(const T* o4)
{
    return (double)o4[0] + (double)o4[1];
}

__device__ __forceinline__ bool finite(double v) { return v == v && v - v == 0.0; }

__device__ void record(dstate* st, double* hist, double rn)
{
    if (hist && st->hist_len < st->hist_cap) {
        hist[2 * st->hist_len] = (double)st->iters;
        hist[2 * st->hist_len + 1] = st->bnorm > 0.0 ? rn / st->bnorm : rn;
        st->hist_len++;
    }
}

// monitor check (default_monitor.h:200-227): converged when the residual is a
// valid number, <= tol and at least min_iters steps ran; finished also at the cap
__device__ void monitor_check(dstate* st, double* hist, double rn)
{
    st->rnorm = rn;
    record(st, hist, rn);
    if (!finite(rn)) {
        st->invalid = 1;
        st->done = 1;
        return;
    }
    if (rn <= st->tol && st->iters >= st->min_iters) {
        st->converged = 1;
        st->done = 1;
        return;
    }
    if (st->iters >= st->max_iters) st->done = 1;
}

// ---------------------------------------------------------------- common kernels

template <typename T>
__global__ void k_init(dstate* st, const T* nb4, double rel_tol, double abs_tol)
{
    const double bn = sqrt(dval(nb4));
    st->bnorm = bn;
    st->tol = abs_tol + rel_tol * bn;
}

// v := s v, s read from device memory
template <typename T>
__global__ __launch_bounds__(DB) void k_scale(size_t n, T* __restrict__ v, const T* __restrict__ s,
                                              const int* __restrict__ skip)
{
    if (*skip) return;
    const T a = *s;
    for (size_t i = (size_t)blockIdx.x * DB + threadIdx.x; i < n; i += (size_t)gridDim.x * DB) v[i] = a * v[i];
}

// y := s x
template <typename T>
__global__ __launch_bounds__(DB) void k_scale_copy(size_t n, const T* __restrict__ x, T* __restrict__ y,
                                                   const T* __restrict__ s, const int* __restrict__ skip)
{
    if (*skip) return;
    const T a = *s;
    for (size_t i = (size_t)blockIdx.x * DB + threadIdx.x; i < n; i += (size_t)gridDim.x * DB) y[i] = a * x[i];
}

template <typename T>
__global__ __launch_bounds__(DB) void k_fill(size_t n, T* __restrict__ v, T a)
{
    for (size_t i = (size_t)blockIdx.x * DB + threadIdx.x; i < n; i += (size_t)gridDim.x * DB) v[i] = a;
}

// max |x_i|: non-negative doubles order like their bit patterns, so blocks fold
// their maxima with one integer atomic max (order-independent)
__global__ __launch_bounds__(DB) void k_absmax(size_t n, const double* __restrict__ x,
                                               unsigned long long* __restrict__ out)
{
    double m = 0.0;
    for (size_t i = (size_t)blockIdx.x * DB + threadIdx.x; i < n; i += (size_t)gridDim.x * DB) m = fmax(m, fabs(x[i]));
    for (int k = 32; k >= 1; k >>= 1) m = fmax(m, __shfl_xor(m, k, 64));
    __shared__ double wm[DB / 64];
    if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < DB / 64; ++w) m = fmax(m, wm[w]);
        atomicMax(out, (unsigned long long)__double_as_longlong(m));
    }
}

// ---------------------------------------------------------------- GMRES kernels

// the power of two 2^-e with |v| 2^-e in [1, 2), within the normal range of T (1 for a
// zero or an invalid v)
template <typename T>
__device__ __forceinline__ double pow2_inverse(double v)
{
    constexpr int lim = sizeof(T) == 8 ? 1000 : 100;
    if (v == 0.0 || !finite(v)) return 1.0;
    const int e = ilogb(v);
    return ldexp(1.0, -(e < -lim ? -lim : e > lim ? lim : e));
}

// restart: beta = ||r||, monitor check on the true residual, g = beta e_1; first (may be
// null): the power of two near 1 / beta
template <typename T, typename S>
__global__ void k_gm_start(dstate* st, const T* n4, double* g, int m, S* sig, T* first, double* hist)
{
    if (st->done) {
        st->stop = 1;
        return;
    }
    const double beta = sqrt(dval(n4));
    monitor_check(st, hist, beta);
    if (st->done) {
        st->stop = 1;
        return;
    }
    st->stop = 0;
    st->cycle_len = 0;
    st->cycles++;
    g[0] = beta;
    for (int i = 1; i <= m; ++i) g[i] = 0.0;
    sig[0] = (S)(1.0 / beta);
    if (first != nullptr) *first = (T)pow2_inverse<T>(beta);
}

__device__ __forceinline__ void apply_rot(double& dx, double& dy, double cs, double sn)
{
    const double t = cs * dx + sn * dy;
    dy = -sn * dx + cs * dy;
    dx = t;
}

// New Hessenberg column j with h_{j+1,j} = hn: previous rotations, new rotation,
// residual estimate (gmres.h:217-274); sig[j+1] = 1 / hn scales the stored basis
// vector (V holds unnormalised vectors; the basis is sig_i V_i).
template <typename T>
__device__ void givens_step(int j, int m, double hn, double* H, int ldh, double* cs, double* sn, double* g, T* sig,
                            dstate* st)
{
    double* Hj = H + (size_t)j * ldh;
    Hj[j + 1] = hn;
    for (int k = 0; k < j; ++k) apply_rot(Hj[k], Hj[k + 1], cs[k], sn[k]);
    double c, s;
    const double dx = Hj[j], dy = Hj[j + 1];
    if (dy == 0.0) {
        c = 1.0;
        s = 0.0;
    } else if (fabs(dy) > fabs(dx)) {
        const double t = dx / dy;
        s = 1.0 / sqrt(1.0 + t * t);
        c = t * s;
    } else {
        const double t = dy / dx;
        c = 1.0 / sqrt(1.0 + t * t);
        s = t * c;
    }
    cs[j] = c;
    sn[j] = s;
    apply_rot(Hj[j], Hj[j + 1], c, s);
    Hj[j + 1] = 0.0;
    apply_rot(g[j], g[j + 1], c, s);
    st->iters++;
    st->cycle_len = j + 1;
    const double est = fabs(g[j + 1]);
    st->rnorm = est;
    sig[j + 1] = hn != 0.0 ? (T)(1.0 / hn) : T(0);
    if (hn == 0.0 || !finite(est) || (st->early_exit && est <= st->tol) || j + 1 >= m || st->iters >= st->max_iters)
        st->stop = 1;
}

template <typename T>
struct basis_pack {
    const T* p[MAXB];
};

// Reductions over many blocks end in per-block totals stored plainly in `part`;
// a one-block kernel launched next merges them in a fixed order (block by block
// per thread, then threads in order) and runs the scalar step.  A last-block ticket
// with relaxed agent-scope stores, as the blocking reductions use up to 256 blocks, needs
// no release, but its increments come one after the other, about 10 ns each: on the 1000
// to 4000 blocks of these grids that is more than the extra launch.
template <typename T, bool COMP>
__device__ __forceinline__ void part_out(T s, T c, T* __restrict__ part, size_t slot)
{
    dev::block_reduce<T, COMP, DB>(s, c);
    if (threadIdx.x == 0) {
        part[2 * slot] = s;
        part[2 * slot + 1] = c;
    }
}

// Per-block totals of N <= 16 sums into slots 0 .. N - 1 of the partials, G apart: one
// transposing reduction per wave, then the waves in order.  One reduction after the other
// costs six dependent merges a sum: with 14 of them (L = 4) the Gram kernel of 872k rows
// spent more on its end than on its reads, 24.7 us, and its merge 21.3.  A whole cycle of
// that solver went from 325 to 297 us with the transposing form on both sides.
template <typename T, bool COMP, int N>
__device__ __forceinline__ void block_totals(const T (&s)[N], const T (&c)[N], T* __restrict__ part)
{
    constexpr int P = N <= 1 ? 1 : N <= 2 ? 2 : N <= 4 ? 4 : N <= 8 ? 8 : 16, NW = DB / 64;
    static_assert(N <= 16, "block_totals");
    T ts[P], tc[P];
#pragma unroll
    for (int k = 0; k < P; ++k) {
        ts[k] = k < N ? s[k] : T(0);
        tc[k] = k < N ? c[k] : T(0);
    }
    dev::wave_reduce_multi<T, COMP, P>(ts, tc);
    __shared__ T ls[NW][P], lc[NW][P];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane % (64 / P) == 0) {
        ls[wid][lane / (64 / P)] = ts[0];
        lc[wid][lane / (64 / P)] = COMP ? tc[0] : T(0);
    }
    __syncthreads();
    if (threadIdx.x < N) {
        T fs = ls[0][threadIdx.x], fc = lc[0][threadIdx.x];
#pragma unroll
        for (int w = 1; w < NW; ++w) {
            if (COMP) dev::merge<T>(fs, fc, ls[w][threadIdx.x], lc[w][threadIdx.x]);
            else fs = fs + ls[w][threadIdx.x];
        }
        const size_t slot = (size_t)threadIdx.x * gridDim.x + blockIdx.x;
        part[2 * slot] = fs;
        part[2 * slot + 1] = fc;
    }
}

// One block of TH threads: columns 0..NQ-1 of G partials each merged (thread t
// takes partials t, t + TH, ... of every column -- independent loads in flight --,
// then the waves' butterflies and the wave totals in order); out valid in thread 0.
template <typename T, bool COMP, int NQ, int TH = DB>
__device__ __forceinline__ void merge_columns(const T* __restrict__ part, unsigned G, double (&out)[NQ])
{
    T fs[NQ], fc[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) fs[q] = fc[q] = T(0);
    for (unsigned b = threadIdx.x; b < G; b += TH) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const T ps = part[2 * ((size_t)q * G + b)];
            const T pc = part[2 * ((size_t)q * G + b) + 1];
            if (COMP) dev::merge<T>(fs[q], fc[q], ps, pc);
            else fs[q] = fs[q] + ps;
        }
    }
    constexpr int P = NQ <= 1 ? 1 : NQ <= 2 ? 2 : NQ <= 4 ? 4 : NQ <= 8 ? 8 : 16;
    T ts[P], tc[P];
#pragma unroll
    for (int k = 0; k < P; ++k) {
        ts[k] = k < NQ ? fs[k] : T(0);
        tc[k] = k < NQ ? fc[k] : T(0);
    }
    dev::wave_reduce_multi<T, COMP, P>(ts, tc);
    constexpr int NW = TH / 64;
    __shared__ T ls[NW][P], lc[NW][P];
    __shared__ double tot[P];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane % (64 / P) == 0) {
        ls[wid][lane / (64 / P)] = ts[0];
        lc[wid][lane / (64 / P)] = COMP ? tc[0] : T(0);
    }
    __syncthreads();
    if (threadIdx.x < NQ) {   // waves merged in wave order
        T s = ls[0][threadIdx.x], c = lc[0][threadIdx.x];
#pragma unroll
        for (int w = 1; w < NW; ++w) {
            if (COMP) dev::merge<T>(s, c, ls[w][threadIdx.x], lc[w][threadIdx.x]);
            else s = s + ls[w][threadIdx.x];
        }
        tot[threadIdx.x] = (double)s + (double)c;
    }
    __syncthreads();
    if (threadIdx.x == 0)
#pragma unroll
        for (int q = 0; q < NQ; ++q) out[q] = tot[q];
}

// One Gram-Schmidt projection pass for column j: per-block partials of
// (V_i, w), i <= j, compensated or plain, KC columns per blockIdx.y chunk;
// k_gm_hfin merges them.  NT: the basis columns are loaded nontemporally (chosen
// when the basis is larger than the 256 MB MALL, so it cannot stay there between
// passes anyway).
template <typename T, int KC, bool COMP, bool NT>
__global__ __launch_bounds__(DB) void k_gm_dot(size_t n, int k, basis_pack<T> V, const T* __restrict__ w,
                                               T* __restrict__ part, const int* __restrict__ stop)
{
    if (*stop) return;
    using Vt = typename dev::vec16<T>::type;   // the vectors come from hipMalloc: 16-byte aligned
    constexpr int W = dev::vec16<T>::W;
    const unsigned G = gridDim.x;
    const int j0 = blockIdx.y * KC;
    const int kc = (k - j0) < KC ? (k - j0) : KC;
    T s[KC], c[KC];
#pragma unroll
    for (int q = 0; q < KC; ++q) s[q] = c[q] = T(0);
    const size_t nv = n / W;
    const Vt* wv = reinterpret_cast<const Vt*>(w);
    for (size_t i = (size_t)blockIdx.x * DB + threadIdx.x; i < nv; i += (size_t)G * DB) {
        const Vt a = wv[i];
#pragma unroll
        for (int q = 0; q < KC; ++q)
            if (q < kc) {
                const Vt* col = reinterpret_cast<const Vt*>(V.p[j0 + q]);
                const Vt v = NT ? dev::load_nt<Vt>(col + i) : col[i];
#pragma unroll
                for (int e = 0; e < W; ++e) {
                    if (COMP) dev::dot2_step<T>(s[q], c[q], dev::vget<T>(v, e), dev::vget<T>(a, e));
                    else s[q] = dev::fma_rn<T>(dev::vget<T>(v, e), dev::vget<T>(a, e), s[q]);
                }
            }
    }
    if (blockIdx.x == 0 && threadIdx.x < n - nv * W) {   // the < W trailing elements
        const size_t i = nv * W + threadIdx.x;
#pragma unroll
        for (int q = 0; q < KC; ++q)
            if (q < kc) {
                if (COMP) dev::dot2_step<T>(s[q], c[q], V.p[j0 + q][i], w[i]);
                else s[q] = dev::fma_rn<T>(V.p[j0 + q][i], w[i], s[q]);
            }
    }
#pragma unroll
    for (int q = 0; q < KC; ++q)
        if (q < kc) part_out<T, COMP>(s[q], c[q], part, (size_t)(j0 + q) * G + blockIdx.x);
}

// h_i = sig_i (V_i, w) from G partials per column: H(i, j) (pass 0) or += (pass 1),
// and coef_i = -h_i sig_i for the update.  One block, a wave per column.
// With kk = k + 1 the last column is (w, w) (pass 0 of the selective
// reorthogonalisation), kept unscaled in st->wn2.
template <typename T, bool COMP>
__global__ __launch_bounds__(1024) void k_gm_hfin(const T* __restrict__ part, unsigned G, int k, int kk,
                                                  const T* __restrict__ sig, double* __restrict__ Hj,
                                                  T* __restrict__ coef, int pass, const int* __restrict__ stop,
                                                  dstate* __restrict__ st)
{
    if (*stop) return;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    for (int col = wid; col < kk; col += 1024 / 64) {
        T fs = T(0), fc = T(0);
        for (unsigned b = lane; b < G; b += 64) {
            const T ps = part[2 * ((size_t)col * G + b)];
            const T pc = part[2 * ((size_t)col * G + b) + 1];
            if (COMP) dev::merge<T>(fs, fc, ps, pc);
            else fs = fs + ps;
        }
        dev::wave_reduce<T, COMP>(fs, fc);
        if (lane == 0) {
            if (col == k) {
                st->wn2 = (double)fs + (double)fc;
                continue;
            }
            const double sg = (double)sig[col];
            const double h = ((double)fs + (double)fc) * sg;
            if (pass == 0) Hj[col] = h;
            else Hj[col] += h;
            coef[col] = (T)(-h * sg);
        }
    }
}

// w += sum_{i<k} coef_i V_i (Dot2 over the terms of each element when COMP), and
// per-block partials of ||w||^2 (compensated) for k_gm_nfin.  NT as in k_gm_dot.
template <typename T, bool COMP, bool NT>
__global__ __launch_bounds__(DB) void k_gm_upd(size_t n, int k, basis_pack<T> V, const T* __restrict__ coef,
                                               T* __restrict__ w, T* __restrict__ part,
                                               const int* __restrict__ skip)
{
    if (*skip) return;
    using Vt = typename dev::vec16<T>::type;
    constexpr int W = dev::vec16<T>::W;
    __shared__ T sc[MAXB];
    for (int q = threadIdx.x; q < k; q += DB) sc[q] = coef[q];
    __syncthreads();
    T ns = T(0), nc = T(0);
    const size_t nv = n / W;
    Vt* wv = reinterpret_cast<Vt*>(w);
    for (size_t i = (size_t)blockIdx.x * DB + threadIdx.x; i < nv; i += (size_t)gridDim.x * DB) {
        Vt a = wv[i];
        T s[W], c[W];
#pragma unroll
        for (int e = 0; e < W; ++e) {
            s[e] = dev::vget<T>(a, e);
            c[e] = T(0);
        }
        for (int q = 0; q < k; ++q) {
            const Vt* col = reinterpret_cast<const Vt*>(V.p[q]);
            const Vt v = NT ? dev::load_nt<Vt>(col + i) : col[i];
            const T cq = sc[q];
#pragma unroll
            for (int e = 0; e < W; ++e) {
                if (COMP) dev::dot2_step<T>(s[e], c[e], cq, dev::vget<T>(v, e));
                else s[e] = dev::fma_rn<T>(cq, dev::vget<T>(v, e), s[e]);
            }
        }
#pragma unroll
        for (int e = 0; e < W; ++e) {
            const T r = COMP ? s[e] + c[e] : s[e];
            reinterpret_cast<T*>(&a)[e] = r;
            if (COMP) dev::dot2_step<T>(ns, nc, r, r);
            else ns = dev::fma_rn<T>(r, r, ns);
        }
        wv[i] = a;
    }
    if (blockIdx.x == 0 && threadIdx.x < n - nv * W) {   // the < W trailing elements
        const size_t i = nv * W + threadIdx.x;
        T s = w[i], c = T(0);
        for (int q = 0; q < k; ++q) {
            if (COMP) dev::dot2_step<T>(s, c, sc[q], V.p[q][i]);
            else s = dev::fma_rn<T>(sc[q], V.p[q][i], s);
        }
        const T r = COMP ? s + c : s;
        w[i] = r;
        if (COMP) dev::dot2_step<T>(ns, nc, r, r);
        else ns = dev::fma_rn<T>(r, r, ns);
    }
    part_out<T, COMP>(ns, nc, part, blockIdx.x);
}

// ||w|| from G partials, then the Givens step for column j with h_{j+1,j} = ||w||
template <typename T, bool COMP>
__global__ __launch_bounds__(DB) void k_gm_nfin(const T* __restrict__ part, unsigned G, int j, int m,
                                                double* __restrict__ H, int ldh, double* __restrict__ cs,
                                                double* __restrict__ sn, double* __restrict__ g, T* __restrict__ sig,
                                                dstate* __restrict__ st, const int* __restrict__ skip)
{
    if (*skip) return;
    double nn[1];
    merge_columns<T, COMP, 1>(part, G, nn);
    if (threadIdx.x == 0) givens_step<T>(j, m, sqrt(nn[0]), H, ldh, cs, sn, g, sig, st);
}

// Selective reorthogonalisation after the first classical pass (Daniel, Gragg,
// Kaufman and Stewart 1976): w' = w - V h is accepted when ||w'|| >= ||w|| / sqrt 2,
// and the Givens step runs with h_{j+1,j} = ||w'||; otherwise the second pass runs
// (skip1 = 0) and k_gm_nfin takes the step after it.
template <typename T, bool COMP>
__global__ __launch_bounds__(DB) void k_gm_dgks(const T* __restrict__ part, unsigned G, int j, int m,
                                                double* __restrict__ H, int ldh, double* __restrict__ cs,
                                                double* __restrict__ sn, double* __restrict__ g, T* __restrict__ sig,
                                                dstate* __restrict__ st)
{
    if (st->stop) {
        if (threadIdx.x == 0) st->skip1 = 1;
        return;
    }
    double nn[1];
    merge_columns<T, COMP, 1>(part, G, nn);
    if (threadIdx.x != 0) return;
    if (nn[0] >= 0.5 * st->wn2) {
        st->skip1 = 1;
        givens_step<T>(j, m, sqrt(nn[0]), H, ldh, cs, sn, g, sig, st);
    } else {
        st->skip1 = 0;
    }
}

// ---- GMRES with delayed reorthogonalisation (gram_schmidt 1).
//
// Classical Gram-Schmidt with two passes, the second one of each vector taken together
// with the first one of the next (Bielich, Langou, Thomas, Swirydowicz, Yamazaki, Boman,
// "Low-synch Gram-Schmidt with delayed reorthogonalization for Krylov solvers", Parallel
// Computing 112, 2022).  Step j holds the final vectors V_i, i < j (basis q_i = sig_i V_i),
// the once-projected candidate u = V_j and z = A u; one pass over the basis takes the
// products of every V_i (and of u itself) with both u and z:
//   s_i = (q_i, u), r_i = (q_i, z);  alpha = sqrt((u, u) - sum s_i^2)  (= h_{j,j-1})
//   q_j = (u - sum s_i q_i) / alpha;  h_{i,j-1} += s_i, i < j (the second projection)
//   t = (q_j, z);  A q_j = (z - sum s_i A q_i) / alpha gives column j of H, and
//   next candidate u' = (z - sum r_i q_i - t q_j) / alpha,
// and one more pass writes V_j and u'.  A step reads the basis twice, where the two
// projections of CGS2 read it four times, and is 4 kernels instead of 8.  Both passes are
// bound by HBM.  128 x 120 x 112 convection-diffusion, FP64 GMRES(30): the kernels of a
// step take 126 us against 226 us with CGS2 (products 41 us = 5.9 TB/s, update 42 us =
// 6.2 TB/s), the whole solve 86.5 ms against 145.4 ms; FP32 inner GMRES(30) in FP64
// refinement on 120 x 128 x 124 60.9 ms against 92.9 ms.  Same steps, same residuals.
// The estimate of step j - 1 is known after the product z = A u of step j; a cycle that
// stops there has formed one z that it does not use.
//
// Scale.  A product of two vectors must neither over- nor underflow where CGS2's (of the
// basis with A q_j) do not, so u and z are kept near 1 and ||A|| by powers of two, which
// change no significand.  V_0 is the residual as it is; step 0 takes z = A (f V_0) with
// f = 2^-e near 1 / ||r|| (k_gm_start).  Its products also hold (z, z), so that
// F = 2^e near ||A q_0|| is known, and every candidate is divided by F: with column j - 1
// completed from such a candidate, s_i and alpha enter H times F.

// Products of the k columns V_0 .. V_{k-1} with u (NV 1) or with u and z (NV 2), over
// chunks of kpc <= 8 columns (blockIdx.y): slot NV i + v of the partials.  FP64 vectors
// take Dot2 steps (COMP); FP32 products are exact in FP64 and are summed there, which is
// more accurate than an FP32 Dot2 and a tenth of its operations.
template <typename T, bool COMP, bool NT, int NV, int KCC>
__device__ __forceinline__ void gm_proj_cols(size_t n, const T* const* __restrict__ cols, const T* __restrict__ u,
                                             const T* __restrict__ z, double (&s)[8 * NV], double (&c)[8 * NV])
{
    using Vt = typename dev::vec16<T>::type;
    constexpr int W = dev::vec16<T>::W;
    constexpr bool D2 = COMP && sizeof(T) == 8;
    const T* p[KCC];
#pragma unroll
    for (int q = 0; q < KCC; ++q) p[q] = cols[q];
    auto step = [&](int q, T v, T a, T b) {
        if constexpr (D2) {
            dev::dot2_step<double>(s[q * NV], c[q * NV], v, a);
            if constexpr (NV == 2) dev::dot2_step<double>(s[q * NV + 1], c[q * NV + 1], v, b);
        } else {
            s[q * NV] = __builtin_fma((double)v, (double)a, s[q * NV]);
            if constexpr (NV == 2) s[q * NV + 1] = __builtin_fma((double)v, (double)b, s[q * NV + 1]);
        }
    };
    const size_t nv = n / W;
    const Vt* uv = reinterpret_cast<const Vt*>(u);
    const Vt* zv = reinterpret_cast<const Vt*>(z);
    for (size_t i = (size_t)blockIdx.x * DB + threadIdx.x; i < nv; i += (size_t)gridDim.x * DB) {
        const Vt a = uv[i];
        Vt b = a;
        if constexpr (NV == 2) b = zv[i];
        Vt v[KCC];
#pragma unroll
        for (int q = 0; q < KCC; ++q) {
            const Vt* col = reinterpret_cast<const Vt*>(p[q]);
            v[q] = NT ? dev::load_nt<Vt>(col + i) : col[i];
        }
#pragma unroll
        for (int q = 0; q < KCC; ++q)
#pragma unroll
            for (int e = 0; e < W; ++e) step(q, dev::vget<T>(v[q], e), dev::vget<T>(a, e), dev::vget<T>(b, e));
    }
    if (blockIdx.x == 0 && threadIdx.x < n - nv * W) {   // the < W trailing elements
        const size_t i = nv * W + threadIdx.x;
        const T a = u[i], b = NV == 2 ? z[i] : a;
#pragma unroll
        for (int q = 0; q < KCC; ++q) step(q, p[q][i], a, b);
    }
}

template <typename T, bool COMP, bool NT, int NV>
__global__ __launch_bounds__(DB) void k_gm_proj(size_t n, int k, int kpc, basis_pack<T> V, const T* __restrict__ u,
                                                const T* __restrict__ z, double* __restrict__ part,
                                                const int* __restrict__ stop)
{
    if (*stop) return;
    constexpr int NS = 8 * NV;
    const int j0 = blockIdx.y * kpc;
    const int kc = (k - j0) < kpc ? (k - j0) : kpc;
    double s[NS], c[NS];
#pragma unroll
    for (int q = 0; q < NS; ++q) s[q] = c[q] = 0.0;
    const T* const* cols = V.p + j0;
    switch (kc) {   // the same in every thread of the block
    case 1: gm_proj_cols<T, COMP, NT, NV, 1>(n, cols, u, z, s, c); break;
    case 2: gm_proj_cols<T, COMP, NT, NV, 2>(n, cols, u, z, s, c); break;
    case 3: gm_proj_cols<T, COMP, NT, NV, 3>(n, cols, u, z, s, c); break;
    case 4: gm_proj_cols<T, COMP, NT, NV, 4>(n, cols, u, z, s, c); break;
    case 5: gm_proj_cols<T, COMP, NT, NV, 5>(n, cols, u, z, s, c); break;
    case 6: gm_proj_cols<T, COMP, NT, NV, 6>(n, cols, u, z, s, c); break;
    case 7: gm_proj_cols<T, COMP, NT, NV, 7>(n, cols, u, z, s, c); break;
    default: gm_proj_cols<T, COMP, NT, NV, 8>(n, cols, u, z, s, c); break;
    }
    dev::wave_reduce_multi<double, true, NS>(s, c);
    constexpr int NW = DB / 64, LG = 64 / NS;
    __shared__ double ls[NW][NS], lc[NW][NS];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane % LG == 0) {
        ls[wid][lane / LG] = s[0];
        lc[wid][lane / LG] = c[0];
    }
    __syncthreads();
    if (threadIdx.x < (unsigned)(kc * NV)) {   // waves merged in wave order
        double fs = ls[0][threadIdx.x], fc = lc[0][threadIdx.x];
#pragma unroll
        for (int w = 1; w < NW; ++w) dev::merge<double>(fs, fc, ls[w][threadIdx.x], lc[w][threadIdx.x]);
        const size_t slot = ((size_t)j0 * NV + threadIdx.x) * gridDim.x + blockIdx.x;
        part[2 * slot] = fs;
        part[2 * slot + 1] = fc;
    }
}

// The scalars of step j from the G partials of each product: column j - 1 of H is
// completed (Givens step, estimate, stop flag) and, unless the cycle ends (LAST, j = m),
// column j of H and the coefficients of k_gm_next are formed.  Hq holds the columns of H
// before the rotations, R after them.  coef: [0, j) of V_j, MAXB + [0, j) of u', then
// u' takes coef[2 MAXB] z + coef[2 MAXB + 1] V_j; coef[2 MAXB + 2] keeps F.  first is f of
// step 0, whose products are those of V_0 and z.  One block: a wave per product for the
// merges, then thread 0 runs the rotations while the waves after the first form column j.
template <typename T, bool LAST>
__global__ __launch_bounds__(1024) void k_gm_step(const double* __restrict__ part, unsigned G, int j,
                                                  double* __restrict__ Hq, double* __restrict__ R, int ldh,
                                                  double* __restrict__ cs, double* __restrict__ sn,
                                                  double* __restrict__ g, double* __restrict__ sig,
                                                  double* __restrict__ coef, const T* __restrict__ first,
                                                  dstate* __restrict__ st)
{
    if (st->stop) return;
    constexpr int NV = LAST ? 1 : 2;
    __shared__ double pr[2 * (MAXB + 1)];           // (V_i, u), (V_i, z); later s_i, r_i
    __shared__ double sg[MAXB], hcol[MAXB + 1], rot[MAXB + 1], lcs[MAXB], lsn[MAXB];
    __shared__ double fac;                          // F
    __shared__ double sca[5];                       // sig_j, t, h_{j,j-1}, sig_j / f, 1 / F
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    if (tid < j) {
        sg[tid] = sig[tid];
        hcol[tid] = Hq[(size_t)(j - 1) * ldh + tid];
        lcs[tid] = tid + 1 < j ? cs[tid] : 0.0;
        lsn[tid] = tid + 1 < j ? sn[tid] : 0.0;
    }
    const int slots = NV * (!LAST && j == 0 ? 2 : j + 1);
    auto merge_slots = [&](auto nc) {   // a wave for N products at a time
        constexpr int N = decltype(nc)::value;
        for (int s0 = wid * N; s0 < slots; s0 += 16 * N) {
            double fs, fc;
            dev::wave_merge_slots<N>(part, G, s0, slots, fs, fc);
            const int slot = s0 + lane / (64 / N);
            if (lane % (64 / N) == 0 && slot < slots) pr[(slot % NV) * (MAXB + 1) + slot / NV] = fs + fc;
        }
    };
    if (slots <= 16) merge_slots(std::integral_constant<int, 1>{});
    else if (slots <= 32) merge_slots(std::integral_constant<int, 2>{});
    else merge_slots(std::integral_constant<int, 4>{});
    __syncthreads();
    double* const s = pr;
    double* const r = pr + MAXB + 1;
    if (tid < j) {
        s[tid] *= sg[tid];
        if (!LAST) r[tid] *= sg[tid];
    }
    __syncthreads();
    if (wid == 0) {
        double ss = 0.0, sr = 0.0;
        for (int i = lane; i < j; i += 64) {
            ss = __builtin_fma(s[i], s[i], ss);
            if (!LAST) sr = __builtin_fma(s[i], r[i], sr);
        }
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) {
            ss += __shfl_xor(ss, m, 64);
            sr += __shfl_xor(sr, m, 64);
        }
        if (lane == 0) {
            const double a2 = s[j] - ss;
            const double al = a2 <= 0.0 ? 0.0 : sqrt(a2);   // a NaN stays one
            double sj = al != 0.0 ? 1.0 / al : 0.0, zf, F;
            if (j == 0) {
                // ||r||^2 out of range: k_gm_start's 1 / ||r||
                if (!(a2 >= 0x1p-900 && a2 <= 0x1p900) && g[0] != 0.0) sj = sig[0];
                zf = sj / (double)*first;
                const double zi = LAST ? 1.0 : pow2_inverse<double>(sqrt(r[1]) * zf);
                F = 1.0 / zi;
                sca[4] = zi;
                coef[2 * MAXB + 2] = F;
            } else {
                zf = sj;
                F = coef[2 * MAXB + 2];
                sca[4] = 1.0 / F;
            }
            sca[0] = sj;
            sca[1] = LAST ? 0.0 : (r[j] - sr) * sj;
            sca[2] = al * F;
            sca[3] = zf;
            fac = F;
        }
    }
    __syncthreads();
    if (tid < j) {
        hcol[tid] = __builtin_fma(s[tid], fac, hcol[tid]);
        Hq[(size_t)(j - 1) * ldh + tid] = hcol[tid];
    }
    if (tid == 0 && j > 0) {
        hcol[j] = sca[2];
        Hq[(size_t)(j - 1) * ldh + j] = sca[2];
    }
    __syncthreads();
    if (tid == 0) {
        sig[j] = sca[0];
        if (j > 0) {
            double dx = hcol[0];
#pragma unroll 4
            for (int i = 0; i + 1 < j; ++i) {
                double dy = hcol[i + 1];
                apply_rot(dx, dy, lcs[i], lsn[i]);
                rot[i] = dx;
                dx = dy;
            }
            const double dy = hcol[j];
            double c, sv;
            if (dy == 0.0) {
                c = 1.0;
                sv = 0.0;
            } else if (fabs(dy) > fabs(dx)) {
                const double t = dx / dy;
                sv = 1.0 / sqrt(1.0 + t * t);
                c = t * sv;
            } else {
                const double t = dy / dx;
                c = 1.0 / sqrt(1.0 + t * t);
                sv = t * c;
            }
            rot[j - 1] = c * dx + sv * dy;
            cs[j - 1] = c;
            sn[j - 1] = sv;
            const double g0 = g[j - 1];
            g[j - 1] = c * g0;
            g[j] = -sv * g0;
            const double est = fabs(sv * g0);
            st->iters++;
            st->cycle_len = j;
            st->rnorm = est;
            if (LAST || sca[2] == 0.0 || !finite(est) || (st->early_exit && est <= st->tol) ||
                st->iters >= st->max_iters)
                st->stop = 1;
        }
    }
    if (!LAST && wid >= 1) {
        const int l = tid - 64;
        const double sj = sca[0], t = sca[1], zf = sca[3], zi = sca[4];
        if (l < j) {
            double h = r[l];
            for (int i = l > 0 ? l - 1 : 0; i + 1 < j; ++i) h = __builtin_fma(-Hq[(size_t)i * ldh + l], s[i], h);
            h = __builtin_fma(-hcol[l], s[j - 1], h);
            Hq[(size_t)j * ldh + l] = h * sj;
            coef[l] = -s[l] * sg[l];
            coef[MAXB + l] = -(sj * zi) * r[l] * sg[l];
        } else if (l == j) {
            Hq[(size_t)j * ldh + j] = (j > 0 ? __builtin_fma(-hcol[j], s[j - 1], t) : t) * zf;
            coef[2 * MAXB] = zf * zi;
            coef[2 * MAXB + 1] = -t * (zf * zi) * sj;
        }
    }
    __syncthreads();
    if (tid < j) R[(size_t)(j - 1) * ldh + tid] = rot[tid];
}

// V_j := u - sum s_i q_i and V_{j+1} := u' (u = V_j and z = V_{j+1} on entry) with the
// coefficients of k_gm_step: Dot2 over the terms of each element when COMP; FP32 vectors
// accumulate their exact products in FP64.
template <typename T, bool COMP, bool NT>
__global__ __launch_bounds__(DB) void k_gm_next(size_t n, int j, basis_pack<T> V, const double* __restrict__ coef,
                                                T* __restrict__ u, T* __restrict__ z, const int* __restrict__ stop)
{
    if (*stop) return;
    using Vt = typename dev::vec16<T>::type;
    constexpr int W = dev::vec16<T>::W;
    constexpr bool D2 = COMP && sizeof(T) == 8;
    __shared__ double cu[MAXB], cz[MAXB];
    for (int q = threadIdx.x; q < j; q += DB) {
        cu[q] = coef[q];
        cz[q] = coef[MAXB + q];
    }
    __syncthreads();
    const double az = coef[2 * MAXB], av = coef[2 * MAXB + 1];
    struct acc_t {
        double us, uc, zs, zc;
    };
    auto begin = [&](acc_t& a, T ue, T ze) {
        a.us = (double)ue;
        a.uc = a.zc = 0.0;
        if constexpr (D2) a.zs = dev::two_prod<double>(az, (double)ze, a.zc);
        else a.zs = az * (double)ze;
    };
    auto add = [&](acc_t& a, double c0, double c1, T v) {
        if constexpr (D2) {
            dev::dot2_step<double>(a.us, a.uc, c0, v);
            dev::dot2_step<double>(a.zs, a.zc, c1, v);
        } else {
            a.us = __builtin_fma(c0, (double)v, a.us);
            a.zs = __builtin_fma(c1, (double)v, a.zs);
        }
    };
    auto end = [&](acc_t& a, T& un, T& zn) {
        un = (T)(D2 ? a.us + a.uc : a.us);
        if constexpr (D2) {
            dev::dot2_step<double>(a.zs, a.zc, av, (double)un);
            zn = (T)(a.zs + a.zc);
        } else {
            zn = (T)__builtin_fma(av, (double)un, a.zs);
        }
    };
    const size_t nv = n / W;
    Vt* uv = reinterpret_cast<Vt*>(u);
    Vt* zv = reinterpret_cast<Vt*>(z);
    for (size_t i = (size_t)blockIdx.x * DB + threadIdx.x; i < nv; i += (size_t)gridDim.x * DB) {
        Vt ue = uv[i], ze = zv[i];
        acc_t a[W];
#pragma unroll
        for (int e = 0; e < W; ++e) begin(a[e], dev::vget<T>(ue, e), dev::vget<T>(ze, e));
        auto load = [&](int q) -> Vt {
            const Vt* col = reinterpret_cast<const Vt*>(V.p[q]);
            return NT ? dev::load_nt<Vt>(col + i) : col[i];
        };
        int q = 0;
        for (; q + 4 <= j; q += 4) {   // four columns' loads in flight
            Vt v[4];
#pragma unroll
            for (int p = 0; p < 4; ++p) v[p] = load(q + p);
#pragma unroll
            for (int p = 0; p < 4; ++p)
#pragma unroll
                for (int e = 0; e < W; ++e) add(a[e], cu[q + p], cz[q + p], dev::vget<T>(v[p], e));
        }
        for (; q < j; ++q) {
            const Vt v = load(q);
#pragma unroll
            for (int e = 0; e < W; ++e) add(a[e], cu[q], cz[q], dev::vget<T>(v, e));
        }
#pragma unroll
        for (int e = 0; e < W; ++e) end(a[e], reinterpret_cast<T*>(&ue)[e], reinterpret_cast<T*>(&ze)[e]);
        uv[i] = ue;
        zv[i] = ze;
    }
    if (blockIdx.x == 0 && threadIdx.x < n - nv * W) {   // the < W trailing elements
        const size_t i = nv * W + threadIdx.x;
        acc_t a;
        begin(a, u[i], z[i]);
        for (int q = 0; q < j; ++q) add(a, cu[q], cz[q], V.p[q][i]);
        end(a, u[i], z[i]);
    }
}

// y = R^{-1} g over the steps of this cycle (gmres.h:204-215); y[k..m) = 0.  One block
// of MAXB threads, row i in thread i: column j's entries are loaded a step ahead, so a
// step costs a division and a barrier (one thread walking R in global memory took
// 70 us for m = 30).
template <typename T, typename S>
__global__ __launch_bounds__(MAXB) void k_gm_backsub(int m, const double* __restrict__ H, int ldh,
                                                     const double* __restrict__ g, const S* __restrict__ sig,
                                                     T* __restrict__ y, const dstate* __restrict__ st)
{
    if (st->done) return;
    const int k = st->cycle_len, i = threadIdx.x;
    __shared__ double piv[2];   // alternating, so that one barrier per step suffices
    double gi = i < k ? g[i] : 0.0;
    double h = (i < k && k > 0) ? H[(size_t)(k - 1) * ldh + i] : 0.0;
    for (int j = k - 1; j >= 0; --j) {
        const double hn = (j > 0 && i < j) ? H[(size_t)(j - 1) * ldh + i] : 0.0;
        if (i == j) {
            gi = gi / h;
            piv[j & 1] = gi;
        }
        __syncthreads();
        if (i < j) gi -= h * piv[j & 1];
        h = hn;
    }
    // x += sum_j g_j (sig_j V_j)
    if (i < m) y[i] = i < k ? (T)(gi * (double)sig[i]) : T(0);
}

// x += sum_{j < cycle_len} y_j V_j (compensated: Dot2 over the terms of each element)
template <typename T, bool COMP>
__global__ __launch_bounds__(DB) void k_gm_xupd(size_t n, basis_pack<T> V, const T* __restrict__ y,
                                                T* __restrict__ x, const dstate* __restrict__ st)
{
    if (st->done) return;
    const int k = st->cycle_len;
    __shared__ T sy[MAXB];
    for (int j = threadIdx.x; j < k; j += DB) sy[j] = y[j];
    __syncthreads();
    for (size_t i = (size_t)blockIdx.x * DB + threadIdx.x; i < n; i += (size_t)gridDim.x * DB) {
        T s = x[i], c = T(0);
        for (int j = 0; j < k; ++j) {
            if (COMP) dev::dot2_step<T>(s, c, sy[j], V.p[j][i]);
            else s = dev::fma_rn<T>(sy[j], V.p[j][i], s);
        }
        x[i] = COMP ? s + c : s;
    }
}

// ---------------------------------------------------------------- BiCGStab(L) kernels

template <typename T>
struct bs_pack {
    T* r[MAXL + 1];
    T* u[MAXL + 1];
};

template <typename T>
__global__ void k_bs_init(dstate* st, const T* n4, T* scal, double* hist)
{
    const double rn = sqrt(dval(n4));
    st->rho = 1.0;
    st->alpha = 0.0;
    st->omega = 1.0;
    monitor_check(st, hist, rn);
    *scal = rn != 0.0 ? (T)(1.0 / rn) : T(1);
}

// rho1 = (r_j, rt); beta = alpha rho1 / rho (bicgstabl.h:199-206)
__device__ __forceinline__ void breakdown_stop(dstate* st)
{
    st->breakdown = 1;
    st->done = 1;
    st->stop = 1;
}

template <typename T>
__global__ void k_bs_beta(dstate* st, const T* d4, T* coef, int first, const int* skip)
{
    if (*skip) return;
    double rho = st->rho;
    if (first) rho = -st->omega * rho;
    if (rho == 0.0 || !finite(rho)) {
        breakdown_stop(st);
        return;
    }
    const double rho1 = dval(d4);
    const double beta = st->alpha * rho1 / rho;
    st->rho = rho1;
    coef[0] = (T)beta;
}

// alpha = rho / (u_{j+1}, rt)
template <typename T>
__global__ void k_bs_alpha(dstate* st, const T* d4, T* coef, const int* skip)
{
    if (*skip) return;
    const double sg = dval(d4);
    if (sg == 0.0 || !finite(sg)) {
        breakdown_stop(st);
        return;
    }
    st->alpha = st->rho / sg;
    coef[1] = (T)st->alpha;
}

// u_i = r_i - beta u_i, i = 0..j
template <typename T>
__global__ __launch_bounds__(DB) void k_bs_upd_u(size_t n, int j, bs_pack<T> P, const T* __restrict__ coef,
                                                 const int* __restrict__ skip)
{
    if (*skip) return;
    const T beta = coef[0];
    for (size_t i = (size_t)blockIdx.x * DB + threadIdx.x; i < n; i += (size_t)gridDim.x * DB)
        for (int q = 0; q <= j; ++q) P.u[q][i] = dev::fma_rn<T>(-beta, P.u[q][i], P.r[q][i]);
}

// r_i -= alpha u_{i+1}, i = 0..j;  x += alpha u_0
template <typename T>
__global__ __launch_bounds__(DB) void k_bs_upd_r(size_t n, int j, bs_pack<T> P, T* __restrict__ x,
                                                 const T* __restrict__ coef, const int* __restrict__ skip)
{
    if (*skip) return;
    const T alpha = coef[1];
    for (size_t i = (size_t)blockIdx.x * DB + threadIdx.x; i < n; i += (size_t)gridDim.x * DB) {
        for (int q = 0; q <= j; ++q) P.r[q][i] = dev::fma_rn<T>(-alpha, P.u[q + 1][i], P.r[q][i]);
        x[i] = dev::fma_rn<T>(alpha, P.u[0][i], x[i]);
    }
}

// MR part: gram[k] holds (r_i, r_k), i = 0..k, as 4-word (s, c, ...) entries.
// Solves G g = c by Cholesky in FP64; coef[2 + j] = g_{j+1}.
template <typename T>
__global__ void k_bs_mr(dstate* st, int L, const T* gram, int gstride, T* coef, const int* skip)
{
    if (*skip) return;
    double G[MAXL][MAXL], c[MAXL], y[MAXL];
    for (int k = 1; k <= L; ++k) {
        const T* gk = gram + (size_t)k * gstride;   // entries (r_i, r_k), i = 0..k
        c[k - 1] = dval(gk);
        for (int i = 1; i <= k; ++i) {
            const double v = dval(gk + 4 * i);
            G[i - 1][k - 1] = v;
            G[k - 1][i - 1] = v;
        }
    }
    // Cholesky G = R^T R (upper R stored in G)
    for (int j = 0; j < L; ++j) {
        double d = G[j][j];
        for (int k = 0; k < j; ++k) d -= G[k][j] * G[k][j];
        if (!(d > 0.0) || !finite(d)) {
            breakdown_stop(st);
            return;
        }
        d = sqrt(d);
        G[j][j] = d;
        for (int i = j + 1; i < L; ++i) {
            double v = G[j][i];
            for (int k = 0; k < j; ++k) v -= G[k][j] * G[k][i];
            G[j][i] = v / d;
        }
    }
    for (int i = 0; i < L; ++i) {   // R^T y = c
        double v = c[i];
        for (int k = 0; k < i; ++k) v -= G[k][i] * y[k];
        y[i] = v / G[i][i];
    }
    for (int i = L - 1; i >= 0; --i) {   // R g = y
        double v = y[i];
        for (int k = i + 1; k < L; ++k) v -= G[i][k] * y[k];
        y[i] = v / G[i][i];
    }
    st->omega = y[L - 1];
    for (int j = 0; j < L; ++j) coef[2 + j] = (T)y[j];
}

// x += sum_j g_j r_{j-1};  r_0 -= sum_j g_j r_j;  u_0 -= sum_j g_j u_j  (j = 1..L)
template <typename T, bool COMP>
__global__ __launch_bounds__(DB) void k_bs_upd_mr(size_t n, int L, bs_pack<T> P, T* __restrict__ x,
                                                  const T* __restrict__ coef, const int* __restrict__ skip)
{
    if (*skip) return;
    __shared__ T gm[MAXL];
    if (threadIdx.x < (unsigned)L) gm[threadIdx.x] = coef[2 + threadIdx.x];
    __syncthreads();
    for (size_t i = (size_t)blockIdx.x * DB + threadIdx.x; i < n; i += (size_t)gridDim.x * DB) {
        T sx = x[i], cx = T(0), sr = P.r[0][i], cr = T(0), su = P.u[0][i], cu = T(0);
        T rprev = sr;
        for (int j = 1; j <= L; ++j) {
            const T g = gm[j - 1];
            const T rj = P.r[j][i];
            const T uj = P.u[j][i];
            if (COMP) {
                dev::dot2_step<T>(sx, cx, g, rprev);
                dev::dot2_step<T>(sr, cr, -g, rj);
                dev::dot2_step<T>(su, cu, -g, uj);
            } else {
                sx = dev::fma_rn<T>(g, rprev, sx);
                sr = dev::fma_rn<T>(-g, rj, sr);
                su = dev::fma_rn<T>(-g, uj, su);
            }
            rprev = rj;
        }
        x[i] = COMP ? sx + cx : sx;
        P.r[0][i] = COMP ? sr + cr : sr;
        P.u[0][i] = COMP ? su + cu : su;
    }
}

// true residual every recalc_freq cycles (bicgstabl.h:247-263)
__global__ void k_bs_recalc_flag(dstate* st)
{
    st->skip_recalc = 1;
    if (st->done) return;
    const int f = st->recalc_freq;
    if (f > 0 && ((st->iters / st->basis + 1) % f) == 0) st->skip_recalc = 0;
}

template <typename T>
__global__ void k_bs_check(dstate* st, const T* n4, double* hist)
{
    if (st->done) return;
    st->iters += st->basis;
    st->cycles++;
    monitor_check(st, hist, sqrt(dval(n4)));
}

// ---- fused BiCGStab(L) cycle: dots ride on the kernels that produce their operands,
// a one-block kernel merges them and runs the scalar step

// scalar steps of bicgstabl.h:199-210 on merged dot products
template <typename T>
__device__ void epi_alpha(dstate* st, double sg, T* coef)
{
    if (sg == 0.0 || !finite(sg)) {
        breakdown_stop(st);
        return;
    }
    st->alpha = st->rho / sg;
    coef[1] = (T)st->alpha;
}
template <typename T>
__device__ void epi_beta(dstate* st, double rho1, int first, T* coef)
{
    double rho = st->rho;
    if (first) rho = -st->omega * rho;
    if (rho == 0.0 || !finite(rho)) {
        breakdown_stop(st);
        return;
    }
    coef[0] = (T)(st->alpha * rho1 / rho);
    st->rho = rho1;
}

enum { EPI_NONE = 0, EPI_ALPHA, EPI_BETA, EPI_CHECK, EPI_REL };

// end of a cycle: d0 = (r_0, r~), d1 = (r_0, r_0)
template <typename T>
__device__ void epi_cycle(int kind, dstate* st, double d0, double d1, T* coef, double* hist, double delta)
{
    st->iters += st->basis;
    st->cycles++;
    const double rn = sqrt(d1) * st->rscale;
    if (kind == EPI_CHECK) {
        monitor_check(st, hist, rn);
        if (st->done) {
            st->stop = 1;
            return;
        }
    } else {   // reliable updates: pause for an FP64 update, or continue
        st->rnorm = rn;
        if (!finite(rn)) {
            st->invalid = 1;
            st->done = 1;
            st->stop = 1;
            return;
        }
        if (rn <= delta * st->rlast || rn <= st->tol || st->iters >= st->max_iters) {
            st->stop = 1;
            return;
        }
    }
    epi_beta<T>(st, d0, 1, coef);
}

// number of dot products a fused kernel hands to k_ds_fin for step EPI
template <int EPI> struct epi_terms {
    static constexpr int value = EPI == EPI_NONE ? 0 : (EPI == EPI_ALPHA || EPI == EPI_BETA ? 1 : 2);
};

// y = A x (MODE 0) or y = b - A x (MODE 1), LPR lanes per row (Dot2 rows when
// CROWS), rows formed from staged tiles (STAGED) or read by their lanes, with partials of the dot products of y that the cycle needs next
// (k_ds_fin then runs the step):
//   EPI_ALPHA  (y, r~) -> alpha;  EPI_BETA (y, r~) -> beta of the next BiCG step;
//   EPI_CHECK / EPI_REL (y, r~), (y, y) -> monitor check and beta of the next cycle.
template <typename T, int LPR, bool STAGED, bool CROWS, bool COMP, int MODE, int EPI>
__global__ __launch_bounds__(DB) void k_ds_spmv(int rows, int tile, const int* __restrict__ rp, const int* __restrict__ col,
                                                const T* __restrict__ val, const T* __restrict__ x,
                                                const T* __restrict__ b, T* __restrict__ y, const T* __restrict__ rt,
                                                T* __restrict__ part, const int* __restrict__ skip)
{
    if (*skip) return;
    constexpr int NQ = epi_terms<EPI>::value;
    T ds[NQ > 0 ? NQ : 1], dc[NQ > 0 ? NQ : 1];
#pragma unroll
    for (int q = 0; q < (NQ > 0 ? NQ : 1); ++q) ds[q] = dc[q] = T(0);
    const int lane = threadIdx.x % LPR;
    // one row: its lanes accumulate (staged: from the tile in LDS), merge, and lane 0
    // stores y_r and takes the dot products
    auto row = [&](long r, int beg, int end, const T* sv, const T* sx) {
        const T rtr = (NQ >= 1 && lane == 0) ? rt[r] : T(0);   // issued with the row bounds
        T s = T(0), c = T(0);
        if (MODE == 1 && lane == 0) s = b[r];
        if (sv != nullptr) dev::csr_row_acc_staged<T, LPR, CROWS, MODE == 1>(beg, end, lane, sv, sx, s, c);
        else dev::csr_row_acc<T, LPR, CROWS, MODE == 1>(beg, end, lane, col, val, x, s, c);
#pragma unroll
        for (int m = LPR / 2; m >= 1; m >>= 1) {
            const T s2 = __shfl_xor(s, m, 64);
            if (CROWS) {
                const T c2 = __shfl_xor(c, m, 64);
                dev::merge<T>(s, c, s2, c2);
            } else {
                s = s + s2;
            }
        }
        if (lane == 0) {
            const T v = CROWS ? s + c : s;
            y[r] = v;
            if constexpr (NQ >= 1) {
                if (COMP) dev::dot2_step<T>(ds[0], dc[0], v, rtr);
                else ds[0] = dev::fma_rn<T>(v, rtr, ds[0]);
            }
            if constexpr (NQ >= 2) {
                if (COMP) dev::dot2_step<T>(ds[1], dc[1], v, v);
                else ds[1] = dev::fma_rn<T>(v, v, ds[1]);
            }
        }
    };
    if constexpr (STAGED) {   // tiles of 128 rows at up to 4 lanes per row, of tile rows beyond
        constexpr int RT = 128, CAP = LPR <= 4 ? 1024 : 2048;
        __shared__ dev::csr_stage<T, RT, CAP> S;
        const int tr = LPR <= 4 ? RT : tile;
        const dev::xcd_rows R = dev::xcd_rows::of(rows, tr);
        for (long r0 = R.first; r0 < R.end; r0 += R.stride) {
            const int nr = (int)((R.end - r0) < tr ? (R.end - r0) : tr);
            const bool staged = dev::csr_stage_tile<T, RT, CAP, DB>(S, r0, nr, rp, col, val, x);
            const int e0 = staged ? S.rp[0] : 0;
            for (int rr = threadIdx.x / LPR; rr < nr; rr += DB / LPR)
                row(r0 + rr, S.rp[rr] - e0, S.rp[rr + 1] - e0, staged ? S.v : nullptr, S.x);
            __syncthreads();   // the next tile overwrites S
        }
    } else {
        const dev::xcd_rows R = dev::xcd_rows::of(rows, DB / LPR);
        for (long r = R.first + (long)threadIdx.x / LPR; r < R.end; r += R.stride)
            row(r, rp[r], rp[r + 1], nullptr, nullptr);
    }
    if constexpr (NQ > 0) {
        block_totals<T, COMP, NQ>(ds, dc, part);
    }
}

// The same on the sliced-diagonal form of the matrix (hpb_sdia.hpp): a wave per slice of
// 64 rows, four consecutive slices per block; MODE 0 scales y by *dalpha (GMRES with
// selective reorthogonalisation; null: 1).  Bound by HBM or, where the matrix fits, by
// the MALL.  7-point rows, CSR product of the same rows in brackets, us: FP64 1.72 M rows
// 19.1 (37.1), 0.87 M rows 11.2 (20.8), 16.8 M rows 229 (317); FP32 1.90 M rows 14.0
// (29.9), 16.8 M rows 116 (234).  NT: the values are loaded nontemporally, chosen when
// the form is larger than the 256 MB MALL (16.8 M rows FP64 / FP32 229 / 116 us against
// 247 / 144; 1.72 M rows, 113 MB of values: 24.1 against 19.1).
template <typename T, bool CROWS, bool COMP, int MODE, int EPI, bool NT, int NC>
__global__ __launch_bounds__(DB) void k_sd_spmv(int rows, sdia_view<T> A, const T* __restrict__ x,
                                                const T* __restrict__ b, T* __restrict__ y, const T* __restrict__ rt,
                                                T* __restrict__ part, const int* __restrict__ skip,
                                                const T* __restrict__ dalpha)
{
    if (skip != nullptr && *skip) return;
    constexpr int NQ = epi_terms<EPI>::value;
    const T alpha = dalpha != nullptr ? *dalpha : T(1);
    T ds[NQ > 0 ? NQ : 1], dc[NQ > 0 ? NQ : 1];
#pragma unroll
    for (int q = 0; q < (NQ > 0 ? NQ : 1); ++q) ds[q] = dc[q] = T(0);
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long nsl = ((long)rows + 63) >> 6;
    const dev::xcd_rows R = dev::xcd_rows::of(nsl, DB / 64);
    for (long sl0 = R.first; sl0 < R.end; sl0 += R.stride) {
        const long sl = sl0 + wid;
        if (sl >= R.end) break;   // the same in every lane of the wave
        const long r = sl * 64 + lane;
        const bool in = r < rows;
        const long ra = in ? r : rows - 1;
        const T rtr = NQ >= 1 ? rt[ra] : T(0);
        T s = MODE == 1 ? b[ra] : T(0), c = T(0);
        sd::row<T, CROWS, MODE == 1, NT, 0, NC>(A, sl, ra, x, s, c);
        if (in) {
            T v = CROWS ? s + c : s;
            if (alpha != T(1)) v = alpha * v;
            y[r] = v;
            if constexpr (NQ >= 1) {
                if (COMP) dev::dot2_step<T>(ds[0], dc[0], v, rtr);
                else ds[0] = dev::fma_rn<T>(v, rtr, ds[0]);
            }
            if constexpr (NQ >= 2) {
                if (COMP) dev::dot2_step<T>(ds[1], dc[1], v, v);
                else ds[1] = dev::fma_rn<T>(v, v, ds[1]);
            }
        }
    }
    if constexpr (NQ > 0) {
        block_totals<T, COMP, NQ>(ds, dc, part);
    }
}

// merged dot products of a fused kernel (G partials per term), then its scalar step
template <typename T, bool COMP, int EPI>
__global__ __launch_bounds__(FB) void k_ds_fin(const T* __restrict__ part, unsigned G, dstate* __restrict__ st,
                                               T* __restrict__ coef, double* hist, double delta,
                                               const int* __restrict__ skip)
{
    if (*skip) return;
    constexpr int NQ = epi_terms<EPI>::value;
    double out[NQ];
    merge_columns<T, COMP, NQ, FB>(part, G, out);
    if (threadIdx.x != 0) return;
    if (EPI == EPI_ALPHA) epi_alpha<T>(st, out[0], coef);
    else if (EPI == EPI_BETA) epi_beta<T>(st, out[0], 0, coef);
    else epi_cycle<T>(EPI, st, out[0], out[NQ - 1], coef, hist, delta);
}

// MR part in one pass: partials of (r_0, r_k) and (r_i, r_k), 1 <= i <= k <= L;
// k_ds_gfin solves the normal equations by Cholesky in FP64 (as k_bs_mr); L <= 4.
template <typename T, int L, bool COMP>
__global__ __launch_bounds__(DB) void k_ds_gram(size_t n, bs_pack<T> P, T* __restrict__ part,
                                                const int* __restrict__ skip)
{
    if (*skip) return;
    constexpr int NP = L + L * (L + 1) / 2;
    T s[NP], c[NP];
#pragma unroll
    for (int q = 0; q < NP; ++q) s[q] = c[q] = T(0);
    for (size_t i = (size_t)blockIdx.x * DB + threadIdx.x; i < n; i += (size_t)gridDim.x * DB) {
        T r[L + 1];
#pragma unroll
        for (int k = 0; k <= L; ++k) r[k] = P.r[k][i];
        int q = 0;
#pragma unroll
        for (int k = 1; k <= L; ++k) {
#pragma unroll
            for (int i2 = 0; i2 <= k; ++i2) {
                if (COMP) dev::dot2_step<T>(s[q], c[q], r[i2], r[k]);
                else s[q] = dev::fma_rn<T>(r[i2], r[k], s[q]);
                ++q;
            }
        }
    }
    block_totals<T, COMP, NP>(s, c, part);
}

// the Gram matrix and right-hand side from Gp partials per entry, then Cholesky
template <typename T, int L, bool COMP>
__global__ __launch_bounds__(FB) void k_ds_gfin(const T* __restrict__ part, unsigned Gp, dstate* __restrict__ st,
                                                T* __restrict__ coef, const int* __restrict__ skip)
{
    if (*skip) return;
    constexpr int NP = L + L * (L + 1) / 2;
    double out[NP];
    merge_columns<T, COMP, NP, FB>(part, Gp, out);
    if (threadIdx.x != 0) return;
    double G[L][L], cv[L], yv[L];   // every loop unrolled: in registers
    int q = 0;
#pragma unroll
    for (int k = 1; k <= L; ++k)
#pragma unroll
        for (int i2 = 0; i2 <= k; ++i2) {
            const double v = out[q++];
            if (i2 == 0) cv[k - 1] = v;
            else {
                G[i2 - 1][k - 1] = v;
                G[k - 1][i2 - 1] = v;
            }
        }
#pragma unroll
    for (int j = 0; j < L; ++j) {
        double d = G[j][j];
#pragma unroll
        for (int k = 0; k < j; ++k) d -= G[k][j] * G[k][j];
        if (!(d > 0.0) || !finite(d)) {
            breakdown_stop(st);
            return;
        }
        d = sqrt(d);
        G[j][j] = d;
#pragma unroll
        for (int i2 = j + 1; i2 < L; ++i2) {
            double v = G[j][i2];
#pragma unroll
            for (int k = 0; k < j; ++k) v -= G[k][j] * G[k][i2];
            G[j][i2] = v / d;
        }
    }
#pragma unroll
    for (int i2 = 0; i2 < L; ++i2) {
        double v = cv[i2];
#pragma unroll
        for (int k = 0; k < i2; ++k) v -= G[k][i2] * yv[k];
        yv[i2] = v / G[i2][i2];
    }
#pragma unroll
    for (int i2 = L - 1; i2 >= 0; --i2) {
        double v = yv[i2];
#pragma unroll
        for (int k = i2 + 1; k < L; ++k) v -= G[i2][k] * yv[k];
        yv[i2] = v / G[i2][i2];
    }
    st->omega = yv[L - 1];
    for (int j = 0; j < L; ++j) coef[2 + j] = (T)yv[j];
}

// MR update of x, r_0, u_0 (as k_bs_upd_mr) with partials of (r_0, r~), (r_0, r_0)
// of the new r_0; k_ds_fin runs the end-of-cycle step (monitor check or
// reliable-update trigger, beta)
template <typename T, bool COMP>
__global__ __launch_bounds__(DB) void k_ds_upd_mr(size_t n, int L, bs_pack<T> P, T* __restrict__ x,
                                                  const T* __restrict__ rt, const T* __restrict__ coef,
                                                  T* __restrict__ part, const int* __restrict__ skip)
{
    if (*skip) return;
    __shared__ T gm[MAXL];
    if (threadIdx.x < (unsigned)L) gm[threadIdx.x] = coef[2 + threadIdx.x];
    __syncthreads();
    T ds[2] = {T(0), T(0)}, dc[2] = {T(0), T(0)};
    for (size_t i = (size_t)blockIdx.x * DB + threadIdx.x; i < n; i += (size_t)gridDim.x * DB) {
        T sx = x[i], cx = T(0), sr = P.r[0][i], cr = T(0), su = P.u[0][i], cu = T(0);
        T rprev = sr;
        for (int j = 1; j <= L; ++j) {
            const T g = gm[j - 1];
            const T rj = P.r[j][i];
            const T uj = P.u[j][i];
            if (COMP) {
                dev::dot2_step<T>(sx, cx, g, rprev);
                dev::dot2_step<T>(sr, cr, -g, rj);
                dev::dot2_step<T>(su, cu, -g, uj);
            } else {
                sx = dev::fma_rn<T>(g, rprev, sx);
                sr = dev::fma_rn<T>(-g, rj, sr);
                su = dev::fma_rn<T>(-g, uj, su);
            }
            rprev = rj;
        }
        const T r0 = COMP ? sr + cr : sr;
        x[i] = COMP ? sx + cx : sx;
        P.r[0][i] = r0;
        P.u[0][i] = COMP ? su + cu : su;
        if (COMP) {
            dev::dot2_step<T>(ds[0], dc[0], r0, rt[i]);
            dev::dot2_step<T>(ds[1], dc[1], r0, r0);
        } else {
            ds[0] = dev::fma_rn<T>(r0, rt[i], ds[0]);
            ds[1] = dev::fma_rn<T>(r0, r0, ds[1]);
        }
    }
    block_totals<T, COMP, 2>(ds, dc, part);
}

// ---- reliable updates (FP32 iterations, FP64 solution and true residual)

// after a cycle: the FP32 recursive residual decides whether the FP64 solution is
// updated now (reduction by delta since the last update, tolerance reached, or the
// iteration cap); stop pauses the cycle graph until the host ran the update
template <typename T>
__global__ void k_rel_check(dstate* st, const T* n4, double delta)
{
    if (st->stop) return;
    st->iters += st->basis;
    st->cycles++;
    const double rn = sqrt(dval(n4)) * st->rscale;
    st->rnorm = rn;
    if (!finite(rn)) {
        st->invalid = 1;
        st->done = 1;
        st->stop = 1;
        return;
    }
    if (rn <= delta * st->rlast || rn <= st->tol || st->iters >= st->max_iters) st->stop = 1;
}

// x64 += xscale x32, x32 = 0
__global__ __launch_bounds__(DB) void k_rel_flush(size_t n, float* __restrict__ x32, double* __restrict__ x64,
                                                  const dstate* __restrict__ st, const int* __restrict__ skip)
{
    if (*skip) return;
    const double g = st->xscale;
    for (size_t i = (size_t)blockIdx.x * DB + threadIdx.x; i < n; i += (size_t)gridDim.x * DB) {
        x64[i] += g * (double)x32[i];
        x32[i] = 0.0f;
    }
}

// the FP64 true residual norm: monitor check, new reference for delta, resume.
// When the update did not lower the true residual the FP32 recurrences have lost
// their accuracy: the iteration restarts from the new residual (r~, u_0, rho,
// alpha, omega as at the start).
// On a (re)start the FP32 residual scale becomes the power of two at or below ||r||:
// the FP32 iteration then runs on the same significands with exponents near 0,
// and with the matrix scaled to |a_ij| < 1 (mscale) A^L r cannot overflow.
__global__ void k_rel_after(dstate* st, const double* n4, double* hist, int first, double mscale)
{
    if (st->done) return;
    const double rn = sqrt(dval(n4));
    if (first && rn > 0.0 && finite(rn)) {
        st->rscale = ldexp(1.0, ilogb(rn));
        st->xscale = st->rscale * mscale;
    }
    st->restart = first || !(rn < st->rlast);
    st->rlast = rn;
    monitor_check(st, hist, rn);
    if (st->restart) {
        st->rho = 1.0;
        st->alpha = 0.0;
        st->omega = 1.0;
    }
    st->stop = st->done;
}

// a breakdown of the FP32 iteration (rho = 0, or a Gram matrix that is not
// numerically positive definite) in a reliable-update solve: clear the stop flags
// so that an FP64 update and a restart from the true residual follow
__global__ void k_rel_resume(dstate* st)
{
    st->breakdown = 0;
    st->done = 0;
    st->stop = 0;
}

// r32 = (float) r64; on a restart also r~ = r32 / ||r32|| and u_0 = 0
__global__ __launch_bounds__(DB) void k_rel_convert(size_t n, const double* __restrict__ r64, float* __restrict__ r32,
                                                    float* __restrict__ rt, float* __restrict__ u0,
                                                    const dstate* __restrict__ st)
{
    if (st->done) return;
    const double inv = st->rlast > 0.0 ? 1.0 / st->rlast : 1.0;
    const double rs = 1.0 / st->rscale;   // a power of two: exact
    const bool restart = st->restart != 0;
    for (size_t i = (size_t)blockIdx.x * DB + threadIdx.x; i < n; i += (size_t)gridDim.x * DB) {
        const float v = (float)(r64[i] * rs);
        r32[i] = v;
        if (restart) {
            rt[i] = (float)(r64[i] * inv);
            u0[i] = 0.0f;
        }
    }
}

// ---------------------------------------------------------------- host side

double now_s()
{
    return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

template <typename T>
struct dbuf {
    T* p = nullptr;
    dbuf() = default;
    dbuf(const dbuf&) = delete;
    dbuf& operator=(const dbuf&) = delete;
    dbuf(dbuf&& o) noexcept : p(o.p) { o.p = nullptr; }
    ~dbuf() { release(); }
    void release()
    {
        if (p) (void)hipFree(p);
        p = nullptr;
    }
    int alloc(size_t count)
    {
        release();
        const hipError_t e = hipMalloc((void**)&p, sizeof(T) * (count ? count : 1));
        if (e != hipSuccess) return hip_status(e, __FILE__, __LINE__, "device solver workspace");
        return HPB_OK;
    }
};

struct graph_guard {
    hipGraph_t g = nullptr;
    hipGraphExec_t e = nullptr;
    graph_guard() = default;
    graph_guard(const graph_guard&) = delete;
    graph_guard& operator=(const graph_guard&) = delete;
    ~graph_guard() { release(); }
    void release()
    {
        if (e) (void)hipGraphExecDestroy(e);
        if (g) (void)hipGraphDestroy(g);
        e = nullptr;
        g = nullptr;
    }
};

// grid of the streaming vector kernels: up to 8 blocks per CU
unsigned vgrid(const hpb_handle_s* h, size_t n, size_t per_cu = 8)
{
    size_t g = (n + DB - 1) / DB;
    const size_t cap = (size_t)(h->num_cu > 0 ? h->num_cu : 256) * per_cu;
    if (g > cap) g = cap;
    return (unsigned)(g < 1 ? 1 : g);
}
// vector kernels that also leave per-block partials: 4 blocks per CU stream as
// fast and halve what the finishing kernel merges
unsigned rgrid(const hpb_handle_s* h, size_t n) { return vgrid(h, n, 4); }

#define DS_CHECK(call)                  \
    do {                                \
        const int _rc = (call);         \
        if (_rc != HPB_OK) return _rc;  \
    } while (0)

template <typename T>
struct problem {
    hpb_handle_t h;
    int rows;
    int64_t nnz;
    const int* rp;
    const int* ci;
    const T* val;
    const T* b;
    T* x;
};

template <typename T>
int end_capture(hipStream_t st, graph_guard& gg, int rc)
{
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(st, &g);
    if (rc != HPB_OK) {
        if (g) (void)hipGraphDestroy(g);
        return rc;
    }
    if (e != hipSuccess) return hip_status(e, __FILE__, __LINE__, "hipStreamEndCapture");
    gg.g = g;
    HPB_HIP(hipGraphInstantiate(&gg.e, gg.g, nullptr, nullptr, 0));
    return HPB_OK;
}

// multi-dot / multi-update over more than 64 columns: chunks of 64
template <typename T>
int multidot_chunks(hpb_handle_t h, int k, T* const* V, size_t n, const T* w, bool comp, T* d4, const int* skip)
{
    for (int c0 = 0; c0 < k; c0 += HPB_MAX_MULTIDOT) {
        const int kc = k - c0 < HPB_MAX_MULTIDOT ? k - c0 : HPB_MAX_MULTIDOT;
        DS_CHECK(multidot_async<T>(h, kc, (const T* const*)(V + c0), n, w, comp, d4 + 4 * c0, skip));
    }
    return HPB_OK;
}
template <typename T>
int multiaxpy_chunks(hpb_handle_t h, int k, const T* coef, T* const* V, size_t n, T* y, bool comp, const int* skip)
{
    for (int c0 = 0; c0 < k; c0 += HPB_MAX_MULTIDOT) {
        const int kc = k - c0 < HPB_MAX_MULTIDOT ? k - c0 : HPB_MAX_MULTIDOT;
        DS_CHECK(multiaxpy_devcoef<T>(h, kc, coef + c0, (const T* const*)(V + c0), n, y, comp, skip));
    }
    return HPB_OK;
}

template <typename T>
int read_state(hpb_handle_t h, const dstate* d, dstate* out)
{
    HPB_HIP(hipMemcpyAsync(h->hres, d, sizeof(dstate), hipMemcpyDeviceToHost, h->stream));
    HPB_HIP(hipStreamSynchronize(h->stream));
    std::memcpy(out, h->hres, sizeof(dstate));
    return HPB_OK;
}

template <typename T>
int init_state(hpb_handle_t h, dstate* d, const hpb_solver_params& p, int basis, int hist_cap)
{
    dstate s{};
    s.rscale = 1.0;
    s.xscale = 1.0;
    s.max_iters = p.max_iters;
    s.min_iters = p.min_iters;
    s.recalc_freq = p.resid_recalc_freq;
    s.early_exit = p.early_exit;
    s.basis = basis;
    s.hist_cap = hist_cap;
    std::memcpy(h->hres, &s, sizeof s);
    HPB_HIP(hipMemcpyAsync(d, h->hres, sizeof s, hipMemcpyHostToDevice, h->stream));
    HPB_HIP(hipStreamSynchronize(h->stream));
    return HPB_OK;
}

// One solver instance: buffers and the captured cycle graph live as long as the
// object, so repeated solves with the same operands (the inner solves of
// iterative refinement) replay the graph without allocating or capturing again.
// FP64 side of the reliable-update mode: the FP32 iteration runs on P (FP32
// values, right-hand side slot unused, x = the FP32 increment), the FP64 solution
// x64 and true residual b64 - A64 x64 are updated every time the FP32 recursive
// residual has dropped by delta.
struct rel64 {
    const double* val;
    const double* b;
    double* x;
    double delta;
    double mscale;   // the FP32 values are mscale * val (a power of two)
};

template <typename T>
class dsolver : public dsolver_base {
public:
    problem<T> P{};
    hpb_solver_params prm{};
    double target = 0.0;
    int hcap = 0;
    bool reliable = false;
    rel64 R{};

    // target_tol: the relative tolerance of all the runs together
    int setup(const problem<T>& pr, const hpb_solver_params& p, int hist_cap, double target_tol,
              const rel64* rel = nullptr)
    {
        P = pr;
        prm = p;
        target = target_tol;
        hcap = hist_cap;
        reliable = rel != nullptr;
        if (rel) R = *rel;
        DS_CHECK(plan_sdia());
        int rc = prepare();
        if (rc != HPB_OK && A.K > 0) {   // the form is optional: without it a solve may fit
            A = sdia_view<T>{};
            slab.release();
            gg.release();
            HPB_CLEAR_STALE();
            rc = prepare();
        }
        return rc;
    }
    // the workspaces and the captured cycle, with the sliced-diagonal form if A.K > 0
    int prepare()
    {
        DS_CHECK(dst.alloc(1));
        if (hcap) DS_CHECK(dhist.alloc(2 * (size_t)hcap));
        if (reliable) {
            DS_CHECK(r64.alloc((size_t)P.rows));
            DS_CHECK(n4d.alloc(4));
        }
        return prm.solver == HPB_SOLVER_GMRES ? setup_gmres() : setup_bicgstabl();
    }
    bool matches(const problem<T>& pr, const hpb_solver_params& p, int hist_cap) const
    {
        const bool same_problem = pr.h == P.h && pr.rows == P.rows && pr.nnz == P.nnz && pr.rp == P.rp &&
                                  pr.ci == P.ci && pr.val == P.val && pr.b == P.b && pr.x == P.x;
        const bool same_params = p.solver == prm.solver && p.restart == prm.restart && p.basis == prm.basis &&
                                 p.high_precision == prm.high_precision &&
                                 p.compensated_spmv == prm.compensated_spmv && p.gram_schmidt == prm.gram_schmidt &&
                                 p.resid_recalc_freq == prm.resid_recalc_freq;
        return same_problem && same_params && hist_cap == hcap;
    }
    // monitor settings (tolerances, iteration caps, early exit, recalculation)
    // are read from p on every run; the captured graph does not depend on them
    int run(const hpb_solver_params& p, dstate* out)
    {
        prm.max_iters = p.max_iters;
        prm.min_iters = p.min_iters;
        prm.rel_tol = p.rel_tol;
        prm.abs_tol = p.abs_tol;
        prm.early_exit = p.early_exit;
        prm.resid_recalc_freq = p.resid_recalc_freq;
        DS_CHECK(init_state<T>(P.h, dst.p, prm, prm.solver == HPB_SOLVER_GMRES ? 1 : prm.basis, hcap));
        if (reliable) return run_reliable(out);
        return prm.solver == HPB_SOLVER_GMRES ? run_gmres(out) : run_bicgstabl(out);
    }
    const double* history() const { return dhist.p; }

private:
    dbuf<dstate> dst;
    dbuf<double> dhist;
    graph_guard gg;
    dbuf<char> slab;             // the vectors of length rows and the sliced-diagonal form
    std::vector<T*> V, U;
    T* rt = nullptr;             // shadow residual of BiCGStab(L)
    dbuf<double> H, Hq, cs, sn, g, dcoef, dsig;
    sdia_view<T> A{};            // the sliced-diagonal form; A.K == 0: products run on the CSR arrays
    bool nt_mat = false;         // the form is larger than the MALL
    dbuf<T> d4, n4, coef, y, scal, da, db, gram;
    dbuf<double> r64, n4d;
    int gstride = 0;

    double* hist() { return hcap ? dhist.p : nullptr; }

    // nv + nu vectors of n, every one 256-byte aligned, and the sliced-diagonal form when
    // plan_sdia found one, in one allocation (31 allocations of 14 MB took 8 ms with their
    // releases, one of 430 MB 0.3 ms); U ends with r~.
    int alloc_vectors(size_t n, int nv, int nu)
    {
        const size_t per = 256 / sizeof(T), stride = (n + per - 1) / per * per;
        const size_t vecs = sizeof(T) * stride * (size_t)(nv + nu);
        DS_CHECK(slab.alloc(vecs + form_bytes()));
        T* const v = reinterpret_cast<T*>(slab.p);
        V.resize(nv);
        U.resize(nu);
        for (int j = 0; j < nv; ++j) V[j] = v + stride * (size_t)j;
        for (int j = 0; j < nu; ++j) U[j] = v + stride * (size_t)(nv + j);
        rt = nu > 0 ? U[nu - 1] : nullptr;
        return A.K > 0 ? fill_sdia(slab.p + vecs) : HPB_OK;
    }

    // Whether the sliced-diagonal form is worth its two passes, a copy back and its memory
    // (60 us at 100 k rows of 7 entries, 0.1 ms at 1 M, 0.3 ms at 1 M of 27, and up to 0.6
    // ms more where the allocation leaves the runtime's cache).  Smaller products are bound
    // by their launch in either form, and a solve to a loose tolerance may end after a few:
    // four products per digit are counted on.  Whole solves on rows of 5 to 32 diagonals,
    // sliced against CSR, BiCGStab(2):
    //   to 1e-12, plain, 7 diagonals: 22 k rows +6 %, 27 k +5, 32 k +3, 37 k -2, 45 k -3;
    //   to 1e-10, plain: 33 k rows -3 to +7 %, 50 k -12 to -3, 100 k -20 to -4, 1 M -48 to -11;
    //   compensated: 33 k -3 to +18 %, 70 k -11 to +3, 100 k -14 to +2 (7 diagonals), 150 k
    //     -18 to -5;
    //   to 1e-3, plain: 50 k -2 to +5 %, 70 k -6 to +4, 100 k -10 to 0, 1 M -34 to +1;
    //   to 1e-1: -1 to +14 % at 100 k, -21 to +32 at 1 M.
    bool form_pays() const
    {
        const double each = prm.solver == HPB_SOLVER_GMRES ? 1.0 : 2.0;   // products per iteration
        const double products = std::min(-4.0 * std::log10(std::max(target, 1e-16)), each * prm.max_iters);
        const double rows = P.rows, least = prm.compensated_spmv ? 98304.0 : 34816.0;
        return products >= 12.0 && rows >= least && rows * products >= 1.2e6 * (least / 34816.0);
    }

    // Decides on the sliced-diagonal form of the matrix (hpb_sdia.hpp): A.K > 0 when it
    // fits and pays.
    int plan_sdia()
    {
        hpb_handle_t h = P.h;
        hipStream_t st = h->stream;
        A = sdia_view<T>{};
        if (!form_pays() || P.nnz > (int64_t)SD_MAXK * P.rows) return HPB_OK;
        int* info = reinterpret_cast<int*>(h->dres);
        hipLaunchKernelGGL((k_fill<int>), dim3(1), dim3(DB), 0, st, (size_t)2, info, 0);
        hipLaunchKernelGGL(sd::k_sdia_count, dim3(sdia_grid()), dim3(SD_THREADS), 0, st, slices(), P.rows, P.rp, P.ci, info);
        HPB_LAUNCH_CHECK();
        HPB_HIP(hipMemcpyAsync(h->hres, info, 2 * sizeof(int), hipMemcpyDeviceToHost, st));
        HPB_HIP(hipStreamSynchronize(st));
        const int K = reinterpret_cast<const int*>(h->hres)[0], bad = reinterpret_cast<const int*>(h->hres)[1];
        if (!bad && K >= 1 && 4 * (int64_t)slices() * 64 * K <= 5 * P.nnz + 1024) A.K = K;
        return HPB_OK;
    }

    long slices() const { return ((long)P.rows + 63) / 64; }
    size_t form_slots() const { return (size_t)slices() * (size_t)A.K; }
    size_t form_bytes() const { return form_slots() * (64 * sizeof(T) + sizeof(uint64_t) + sizeof(int)); }
    unsigned sdia_grid() const
    {
        const long cus = P.h->num_cu > 0 ? P.h->num_cu : 256;
        return (unsigned)std::min((slices() + 3) / 4, 8 * cus);
    }

    int fill_sdia(char* at)
    {
        const size_t bv = 64 * sizeof(T) * form_slots(), bm = sizeof(uint64_t) * form_slots();
        A.val = reinterpret_cast<const T*>(at);
        A.mask = reinterpret_cast<const uint64_t*>(at + bv);
        A.off = reinterpret_cast<const int*>(at + bv + bm);
        nt_mat = form_bytes() > (size_t)256 * 1024 * 1024;
        const long cus = P.h->num_cu > 0 ? P.h->num_cu : 256;
        const unsigned lds = (unsigned)((sizeof(T) + sizeof(int)) * 64 * (size_t)A.K);
        hipLaunchKernelGGL((sd::k_sdia_fill<T>), dim3((unsigned)std::min(slices(), 32 * cus)), dim3(64), lds, P.h->stream,
                           slices(), P.rows, A.K, P.rp, P.ci, P.val, const_cast<int*>(A.off),
                           const_cast<uint64_t*>(A.mask), const_cast<T*>(A.val));
        HPB_LAUNCH_CHECK();
        return HPB_OK;
    }

    // y = A x or y = b - A x with the dot products of EPI on the sliced-diagonal form;
    // returns the grid.  Without dots up to 16 blocks per CU, with dots 6 (their
    // partials are merged by one block): us at 4 / 6 / 8 / 16 blocks per CU, 1.72 M rows
    // FP64 19.8 / 20.6 / 21.7 / 19.1 without and 22.0 / 23.1 / 23.8 / 22.2 with one dot,
    // 1.90 M rows FP32 16.7 / 14.3 / 16.1 / 14.0 and 17.3 / 15.3 / 17.8 / 15.9.  A
    // multiple of the XCD count, for the row ranges per XCD.
    template <int MODE, int EPI>
    unsigned sd_spmv(const T* x, const T* b, T* y, const T* rtv, const int* skip, const T* dalpha)
    {
        hpb_handle_t h = P.h;
        const long nsl = ((long)P.rows + 63) / 64, cus = h->num_cu > 0 ? h->num_cu : 256;
        long G = std::min((nsl + DB / 64 - 1) / (DB / 64), (EPI == EPI_NONE ? 16 : 6) * cus);
        G = (G + dev::XCD_COUNT - 1) / dev::XCD_COUNT * dev::XCD_COUNT;
        T* part = reinterpret_cast<T*>(h->part);
        auto go = [&](auto crows, auto compc, auto ntc, auto ncc) {
            constexpr bool CR = decltype(crows)::value, CO = decltype(compc)::value, NTB = decltype(ntc)::value;
            hipLaunchKernelGGL((k_sd_spmv<T, CR, CO && EPI != EPI_NONE, MODE, EPI, NTB, decltype(ncc)::value>),
                               dim3((unsigned)G), dim3(DB), 0, h->stream, P.rows, A, x, b, y, rtv, part, skip, dalpha);
        };
        auto go2 = [&](auto crows, auto compc, auto ncc) {
            if (nt_mat) go(crows, compc, std::true_type{}, ncc);
            else go(crows, compc, std::false_type{}, ncc);
        };
        auto go1 = [&](auto crows, auto ncc) {
            if (prm.high_precision) go2(crows, std::true_type{}, ncc);
            else go2(crows, std::false_type{}, ncc);
        };
        // plain rows: the lanes the CSR product would take
        const double mean = (double)P.nnz / P.rows;
        if (prm.compensated_spmv) go1(std::true_type{}, std::integral_constant<int, 2>{});
        else if (mean <= 8.0) go1(std::false_type{}, std::integral_constant<int, 2>{});
        else if (mean <= 12.0) go1(std::false_type{}, std::integral_constant<int, 4>{});
        else if (mean <= 24.0) go1(std::false_type{}, std::integral_constant<int, 8>{});
        else go1(std::false_type{}, std::integral_constant<int, 16>{});
        return (unsigned)G;
    }

    // y = A x (b null; times *dalpha when given) or y = b - A x
    int apply(const T* x, const T* b, T* y, const int* skip, const T* dalpha = nullptr)
    {
        if (A.K == 0)
            return csr_apply<T>(P.h, P.rows, P.nnz, P.rp, P.ci, P.val, x, b, y, prm.compensated_spmv != 0, skip, dalpha);
        if (b) sd_spmv<1, EPI_NONE>(x, b, y, nullptr, skip, nullptr);
        else sd_spmv<0, EPI_NONE>(x, nullptr, y, nullptr, skip, dalpha);
        HPB_LAUNCH_CHECK();
        return HPB_OK;
    }

    // GMRES with delayed reorthogonalisation (k_gm_step): one restart cycle
    int setup_gmres_delayed()
    {
        hpb_handle_t h = P.h;
        hipStream_t st = h->stream;
        const size_t n = (size_t)P.rows;
        const int m = prm.restart, ldh = m + 1;
        const bool comp = prm.high_precision != 0;
        DS_CHECK(alloc_vectors(n, m + 1, 0));
        basis_pack<T> bp{};
        for (int j = 0; j <= m; ++j) bp.p[j] = V[j];
        DS_CHECK(H.alloc((size_t)ldh * m));
        DS_CHECK(Hq.alloc((size_t)ldh * m));
        DS_CHECK(cs.alloc(m));
        DS_CHECK(sn.alloc(m));
        DS_CHECK(g.alloc(m + 1));
        DS_CHECK(n4.alloc(4));
        DS_CHECK(dcoef.alloc(2 * MAXB + 3));
        DS_CHECK(scal.alloc(1));
        DS_CHECK(y.alloc(m));
        DS_CHECK(dsig.alloc(m + 1));
        dstate* S = dst.p;
        const int* done = &S->done;
        const int* stop = &S->stop;
        double* part = reinterpret_cast<double*>(h->part);
        const size_t part_pairs = h->part_bytes / (2 * sizeof(double));
        const size_t cus = (size_t)(h->num_cu > 0 ? h->num_cu : 256);
        const size_t gvec = (n / dev::vec16<T>::W + DB - 1) / DB;
        const bool nt_basis = (double)(m + 1) * (double)n * sizeof(T) > 256.0 * 1024 * 1024;
        // updates: 8 blocks per CU (4 within 2 % either way, 2 up to 20 % slower)
        const unsigned gupd = (unsigned)std::max<size_t>(1, std::min(gvec, 8 * cus));
        using BT = std::true_type;
        using BF = std::false_type;
        auto flags = [&](auto f) {   // f(compensated, nontemporal basis) with the run's constants
            if (comp) {
                if (nt_basis) f(BT{}, BT{});
                else f(BT{}, BF{});
            } else {
                if (nt_basis) f(BF{}, BT{});
                else f(BF{}, BF{});
            }
        };
        // products of columns 0 .. j with u = V_j (and z = V_{j+1}), merged by k_gm_step
        auto project = [&](int j, auto lastc) {
            constexpr bool LAST = decltype(lastc)::value;
            const int k = !LAST && j == 0 ? 2 : j + 1;   // step 0: (z, z) too
            const int nch = (k + 7) / 8, kpc = (k + nch - 1) / nch;
            // 2 blocks per CU over all chunks: 15 columns of 1.72 M FP64 rows 41.1 us,
            // against 40.5 at 1, 45.3 at 4 and 43.6 at 8; 4 columns 15.9, 18.2, 18.0, 19.0;
            // 30 columns of 1.9 M FP32 rows 42.6, 50.4, 45.3, 46.2
            size_t gd = std::min(gvec, std::max<size_t>(1, 2 * cus / nch));
            gd = std::max<size_t>(1, std::min(gd, part_pairs / (2 * (size_t)k)));
            flags([&](auto compc, auto ntc) {
                constexpr bool C = decltype(compc)::value, NTB = decltype(ntc)::value;
                hipLaunchKernelGGL((k_gm_proj<T, C, NTB, LAST ? 1 : 2>), dim3((unsigned)gd, nch), dim3(DB), 0, st, n,
                                   k, kpc, bp, V[j], LAST ? V[j] : V[LAST ? j : j + 1], part, stop);
            });
            hipLaunchKernelGGL((k_gm_step<T, LAST>), dim3(1), dim3(1024), 0, st, part, (unsigned)gd, j, Hq.p, H.p, ldh,
                               cs.p, sn.p, g.p, dsig.p, dcoef.p, scal.p, S);
        };
        HPB_HIP(hipStreamSynchronize(st));
        HPB_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
        int rc = [&]() -> int {
            DS_CHECK(apply(P.x, P.b, V[0], done));
            DS_CHECK(nrm2_async<T>(h, n, V[0], n4.p, comp, done));
            hipLaunchKernelGGL((k_gm_start<T, double>), dim3(1), dim3(1), 0, st, S, n4.p, g.p, m, dsig.p, scal.p, hist());
            for (int j = 0; j < m; ++j) {
                DS_CHECK(apply(V[j], nullptr, V[j + 1], stop, j == 0 ? scal.p : nullptr));
                project(j, BF{});
                flags([&](auto compc, auto ntc) {
                    constexpr bool C = decltype(compc)::value, NTB = decltype(ntc)::value;
                    hipLaunchKernelGGL((k_gm_next<T, C, NTB>), dim3(gupd), dim3(DB), 0, st, n, j, bp, dcoef.p, V[j],
                                       V[j + 1], stop);
                });
            }
            project(m, BT{});
            hipLaunchKernelGGL((k_gm_backsub<T, double>), dim3(1), dim3(MAXB), 0, st, m, H.p, ldh, g.p, dsig.p, y.p, S);
            if (comp)
                hipLaunchKernelGGL((k_gm_xupd<T, true>), dim3(vgrid(h, n)), dim3(DB), 0, st, n, bp, y.p, P.x, S);
            else
                hipLaunchKernelGGL((k_gm_xupd<T, false>), dim3(vgrid(h, n)), dim3(DB), 0, st, n, bp, y.p, P.x, S);
            return HPB_OK;
        }();
        return end_capture<T>(st, gg, rc);
    }

    // GMRES with selective reorthogonalisation (gram_schmidt 2): the second classical
    // pass of a step runs only when the first one asks for it
    int setup_gmres()
    {
        if (prm.gram_schmidt != 2) return setup_gmres_delayed();
        hpb_handle_t h = P.h;
        hipStream_t st = h->stream;
        const size_t n = (size_t)P.rows;
        const int m = prm.restart;
        const bool comp = prm.high_precision != 0;
        const int ldh = m + 1;
        DS_CHECK(alloc_vectors(n, m + 1, 0));
        DS_CHECK(H.alloc((size_t)ldh * m));
        DS_CHECK(cs.alloc(m));
        DS_CHECK(sn.alloc(m));
        DS_CHECK(g.alloc(m + 1));
        DS_CHECK(n4.alloc(4));
        DS_CHECK(coef.alloc(m + 1));
        DS_CHECK(y.alloc(m));
        DS_CHECK(scal.alloc(m + 1));   // sig_i: the basis is sig_i V_i
        dstate* S = dst.p;
        const int* done = &S->done;
        const int* stop = &S->stop;
        basis_pack<T> bp{};
        for (int j = 0; j <= m; ++j) bp.p[j] = V[j];
        double* hp = hist();
        T* sig = scal.p;
        T* part = reinterpret_cast<T*>(h->part);
        const size_t cus = (size_t)(h->num_cu > 0 ? h->num_cu : 256);
        const size_t part_pairs = h->part_bytes / (2 * sizeof(T));
        // grids over 16-byte vectors; the reductions end in per-block partials
        // merged by one-block kernels (k_gm_hfin, k_gm_nfin)
        const size_t gvec = (n / dev::vec16<T>::W + DB - 1) / DB;
        // basis larger than the 256 MB MALL: stream it (128^3 FP64 GMRES(50), 816 MB:
        // 0.275 s against 0.293 s; 256^3 FP64 GMRES(30): 11.79 s against 12.63 s); a
        // basis that fits is read back from the MALL by the next pass (128^3 FP32
        // GMRES(30), 248 MB: 0.106 s streamed against 0.098 s)
        const bool nt_basis = (double)(m + 1) * (double)n * sizeof(T) > 256.0 * 1024 * 1024;
        // multi-dot blocks per CU over all column chunks: 8 from 2^23 rows (256^3 FP64
        // GMRES(30): 10.99 s, against 11.78 s at 4, 11.10 s at 16), else 4 (128^3:
        // 8 per CU cost 3-6 %, 2 and 1 per CU 2-9 %); updates: 8 per CU (2 and 1 per CU
        // were 4-35 % slower, 16 the same)
        const size_t gd_per_cu = n >= ((size_t)1 << 23) ? 8 : 4;
        const unsigned gupd = (unsigned)std::max<size_t>(1, std::min(gvec, 8 * cus));
        constexpr int KC = 8;
        HPB_HIP(hipStreamSynchronize(st));
        HPB_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
        int rc = [&]() -> int {
            DS_CHECK(apply(P.x, P.b, V[0], done));
            DS_CHECK(nrm2_async<T>(h, n, V[0], n4.p, comp, done));
            hipLaunchKernelGGL((k_gm_start<T, T>), dim3(1), dim3(1), 0, st, S, n4.p, g.p, m, sig, (T*)nullptr, hp);
            for (int j = 0; j < m; ++j) {
                const int k = j + 1;
                // w = A (sig_j V_j), stored unnormalised in V[j+1]
                DS_CHECK(apply(V[j], nullptr, V[j + 1], stop,
                                      sig + j));
                double* Hj = H.p + (size_t)j * ldh;
                for (int pass = 0; pass < 2; ++pass) {
                    // pass 1 runs under skip1 when the first pass may be accepted
                    const int* skip = pass == 1 ? &S->skip1 : stop;
                    const int kk = pass == 0 ? k + 1 : k;   // + (w, w)
                    const unsigned nch = (unsigned)((kk + KC - 1) / KC);
                    size_t gd = std::min(gvec, std::max<size_t>(cus, (gd_per_cu * cus) / nch));
                    gd = std::max<size_t>(1, std::min(gd, part_pairs / (size_t)kk));
                    auto dot = [&](auto compc, auto ntc) {
                        constexpr bool C = decltype(compc)::value, NTB = decltype(ntc)::value;
                        hipLaunchKernelGGL((k_gm_dot<T, KC, C, NTB>), dim3((unsigned)gd, nch), dim3(DB), 0, st, n,
                                           kk, bp, V[j + 1], part, skip);
                        hipLaunchKernelGGL((k_gm_hfin<T, C>), dim3(1), dim3(1024), 0, st, part, (unsigned)gd, k, kk,
                                           sig, Hj, coef.p, pass, skip, S);
                    };
                    auto upd = [&](auto compc) {
                        constexpr bool C = decltype(compc)::value;
                        if (nt_basis)
                            hipLaunchKernelGGL((k_gm_upd<T, C, true>), dim3(gupd), dim3(DB), 0, st, n, k, bp,
                                               coef.p, V[j + 1], part, skip);
                        else
                            hipLaunchKernelGGL((k_gm_upd<T, C, false>), dim3(gupd), dim3(DB), 0, st, n, k, bp,
                                               coef.p, V[j + 1], part, skip);
                        if (pass == 0)
                            hipLaunchKernelGGL((k_gm_dgks<T, C>), dim3(1), dim3(DB), 0, st, part, gupd, j, m, H.p,
                                               ldh, cs.p, sn.p, g.p, sig, S);
                        else
                            hipLaunchKernelGGL((k_gm_nfin<T, C>), dim3(1), dim3(DB), 0, st, part, gupd, j, m, H.p,
                                               ldh, cs.p, sn.p, g.p, sig, S, skip);
                    };
                    using BT = std::true_type;
                    using BF = std::false_type;
                    if (comp) {
                        if (nt_basis) dot(BT{}, BT{});
                        else dot(BT{}, BF{});
                    } else {
                        if (nt_basis) dot(BF{}, BT{});
                        else dot(BF{}, BF{});
                    }
                    if (comp) upd(BT{});
                    else upd(BF{});
                }
            }
            hipLaunchKernelGGL((k_gm_backsub<T, T>), dim3(1), dim3(MAXB), 0, st, m, H.p, ldh, g.p, sig, y.p, S);
            if (comp)
                hipLaunchKernelGGL((k_gm_xupd<T, true>), dim3(vgrid(h, n)), dim3(DB), 0, st, n, bp, y.p, P.x, S);
            else
                hipLaunchKernelGGL((k_gm_xupd<T, false>), dim3(vgrid(h, n)), dim3(DB), 0, st, n, bp, y.p, P.x, S);
            return HPB_OK;
        }();
        return end_capture<T>(st, gg, rc);
    }

    int run_gmres(dstate* out)
    {
        hpb_handle_t h = P.h;
        hipStream_t st = h->stream;
        const bool comp = prm.high_precision != 0;
        DS_CHECK(nrm2_async<T>(h, (size_t)P.rows, P.b, n4.p, comp, nullptr));
        hipLaunchKernelGGL((k_init<T>), dim3(1), dim3(1), 0, st, dst.p, n4.p, prm.rel_tol, prm.abs_tol);
        HPB_LAUNCH_CHECK();
        // every replay starts with the restart residual and the monitor check,
        // so the replay after the last useful cycle ends the solve
        const int max_cycles = prm.max_iters + 2;
        for (int c = 0; c < max_cycles; ++c) {
            HPB_HIP(hipGraphLaunch(gg.e, st));
            DS_CHECK(read_state<T>(h, dst.p, out));
            if (out->done) break;
        }
        return HPB_OK;
    }

    // fused launchers of the BiCGStab(L) cycle (L <= 4, residual recomputed every
    // cycle or never, or reliable updates)
    template <int MODE, int EPI>
    void ds_spmv(const T* x, const T* b, T* y, const T* rtv, const int* skip)
    {
        hpb_handle_t h = P.h;
        if (A.K > 0) {
            const unsigned G = sd_spmv<MODE, EPI>(x, b, y, rtv, skip, nullptr);
            if constexpr (EPI != EPI_NONE) ds_fin<EPI>(G, skip);
            return;
        }
        const double mean = P.rows > 0 ? (double)P.nnz / P.rows : 1.0;
        const int lpr = mean <= 8.0 ? 2 : (mean <= 12.0 ? 4 : (mean <= 24.0 ? 8 : 16));   // as the library SpMV
        // rows of a staged tile beyond 4 lanes, three quarters of its 2048 entries on average
        const int rt = lpr <= 4 || P.nnz < DS_WIDE_NNZ ? 0 : (int)std::min(128.0, 0.75 * 2048 / mean);
        const bool wide = rt >= 4;
        const long per_block = lpr <= 4 ? 128 : wide ? rt : DB / lpr;
        long grid = (P.rows + per_block - 1) / per_block;
        const long cap = (long)(h->num_cu > 0 ? h->num_cu : 256) * 16;   // the gathers want many waves
        grid = std::max(1L, std::min(grid, cap));
        const bool cr = prm.compensated_spmv != 0, comp = prm.high_precision != 0;
        T* part = reinterpret_cast<T*>(h->part);
#define DS_SPMV(L_, ST_, CR_, CO_)                                                                             \
    hipLaunchKernelGGL((k_ds_spmv<T, L_, ST_, CR_, CO_, MODE, EPI>), dim3((unsigned)grid), dim3(DB), 0, h->stream, \
                       P.rows, rt, P.rp, P.ci, P.val, x, b, y, rtv, part, skip)
#define DS_SPMV_L(L_, ST_)                                                                                     \
    do {                                                                                                       \
        if (cr) { if (comp) DS_SPMV(L_, ST_, true, true); else DS_SPMV(L_, ST_, true, false); }                \
        else { if (comp) DS_SPMV(L_, ST_, false, true); else DS_SPMV(L_, ST_, false, false); }                 \
    } while (0)
        if (lpr == 2) DS_SPMV_L(2, true);
        else if (lpr == 4) DS_SPMV_L(4, true);
        else if (lpr == 8 && wide) DS_SPMV_L(8, true);
        else if (lpr == 8) DS_SPMV_L(8, false);
        else if (wide) DS_SPMV_L(16, true);
        else DS_SPMV_L(16, false);
#undef DS_SPMV_L
#undef DS_SPMV
        if constexpr (EPI != EPI_NONE) ds_fin<EPI>((unsigned)grid, skip);
    }

    // the scalar step after a fused kernel whose G blocks left partials in part
    template <int EPI>
    void ds_fin(unsigned G, const int* skip)
    {
        hpb_handle_t h = P.h;
        const T* part = reinterpret_cast<const T*>(h->part);
        if (prm.high_precision)
            hipLaunchKernelGGL((k_ds_fin<T, true, EPI>), dim3(1), dim3(FB), 0, h->stream, part, G, dst.p, coef.p,
                               hist(), R.delta, skip);
        else
            hipLaunchKernelGGL((k_ds_fin<T, false, EPI>), dim3(1), dim3(FB), 0, h->stream, part, G, dst.p, coef.p,
                               hist(), R.delta, skip);
    }

    bool fused_ok() const
    {
        return prm.basis <= 4 && (reliable || prm.resid_recalc_freq == 0 || prm.resid_recalc_freq == 1);
    }

    template <int L>
    void ds_gram(bs_pack<T> bp, const int* skip)
    {
        hpb_handle_t h = P.h;
        const size_t n = (size_t)P.rows;
        T* part = reinterpret_cast<T*>(h->part);
        const unsigned G = rgrid(h, n);
        if (prm.high_precision) {
            hipLaunchKernelGGL((k_ds_gram<T, L, true>), dim3(G), dim3(DB), 0, h->stream, n, bp, part, skip);
            hipLaunchKernelGGL((k_ds_gfin<T, L, true>), dim3(1), dim3(FB), 0, h->stream, part, G, dst.p, coef.p,
                               skip);
        } else {
            hipLaunchKernelGGL((k_ds_gram<T, L, false>), dim3(G), dim3(DB), 0, h->stream, n, bp, part, skip);
            hipLaunchKernelGGL((k_ds_gfin<T, L, false>), dim3(1), dim3(FB), 0, h->stream, part, G, dst.p, coef.p,
                               skip);
        }
    }

    int setup_bicgstabl()
    {
        fused = fused_ok();
        if (fused) return setup_bicgstabl_fused();
        hpb_handle_t h = P.h;
        hipStream_t st = h->stream;
        const size_t n = (size_t)P.rows;
        const int L = prm.basis;
        const bool comp = prm.high_precision != 0;
        DS_CHECK(alloc_vectors(n, L + 1, L + 2));
        bs_pack<T> bp{};
        for (int j = 0; j <= L; ++j) {
            bp.r[j] = V[j];
            bp.u[j] = U[j];
        }
        gstride = 4 * (L + 1);
        DS_CHECK(n4.alloc(4));
        DS_CHECK(da.alloc(4));
        DS_CHECK(db.alloc(4));
        DS_CHECK(gram.alloc((size_t)gstride * (L + 1)));
        DS_CHECK(coef.alloc(2 + MAXL));
        DS_CHECK(scal.alloc(1));
        dstate* S = dst.p;
        // reliable mode pauses the cycle with stop while the host updates x64
        const int* done = reliable ? &S->stop : &S->done;
        const unsigned vg = vgrid(h, n);
        double* hp = hist();
        HPB_HIP(hipStreamSynchronize(st));
        HPB_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
        int rc = [&]() -> int {
            for (int j = 0; j < L; ++j) {
                DS_CHECK(dot2_async<T>(h, n, V[j], rt, da.p, comp, done));
                hipLaunchKernelGGL((k_bs_beta<T>), dim3(1), dim3(1), 0, st, S, da.p, coef.p, j == 0 ? 1 : 0, done);
                hipLaunchKernelGGL((k_bs_upd_u<T>), dim3(vg), dim3(DB), 0, st, n, j, bp, coef.p, done);
                DS_CHECK(apply(U[j], nullptr, U[j + 1], done));
                DS_CHECK(dot2_async<T>(h, n, U[j + 1], rt, db.p, comp, done));
                hipLaunchKernelGGL((k_bs_alpha<T>), dim3(1), dim3(1), 0, st, S, db.p, coef.p, done);
                hipLaunchKernelGGL((k_bs_upd_r<T>), dim3(vg), dim3(DB), 0, st, n, j, bp, P.x, coef.p, done);
                DS_CHECK(apply(V[j], nullptr, V[j + 1], done));
            }
            for (int k = 1; k <= L; ++k)
                DS_CHECK(multidot_async<T>(h, k + 1, (const T* const*)V.data(), n, V[k], comp,
                                           gram.p + (size_t)k * gstride, done));
            hipLaunchKernelGGL((k_bs_mr<T>), dim3(1), dim3(1), 0, st, S, L, gram.p, gstride, coef.p, done);
            if (comp)
                hipLaunchKernelGGL((k_bs_upd_mr<T, true>), dim3(vg), dim3(DB), 0, st, n, L, bp, P.x, coef.p, done);
            else
                hipLaunchKernelGGL((k_bs_upd_mr<T, false>), dim3(vg), dim3(DB), 0, st, n, L, bp, P.x, coef.p, done);
            if (reliable) {
                DS_CHECK(nrm2_async<T>(h, n, V[0], n4.p, comp, done));
                hipLaunchKernelGGL((k_rel_check<T>), dim3(1), dim3(1), 0, st, S, n4.p, R.delta);
                return HPB_OK;
            }
            hipLaunchKernelGGL(k_bs_recalc_flag, dim3(1), dim3(1), 0, st, S);
            DS_CHECK(apply(P.x, P.b, V[0], &S->skip_recalc));
            DS_CHECK(nrm2_async<T>(h, n, V[0], n4.p, comp, done));
            hipLaunchKernelGGL((k_bs_check<T>), dim3(1), dim3(1), 0, st, S, n4.p, hp);
            return HPB_OK;
        }();
        return end_capture<T>(st, gg, rc);
    }

    int setup_bicgstabl_fused()
    {
        hpb_handle_t h = P.h;
        hipStream_t st = h->stream;
        const size_t n = (size_t)P.rows;
        const int L = prm.basis;
        const bool comp = prm.high_precision != 0;
        DS_CHECK(alloc_vectors(n, L + 1, L + 2));
        bs_pack<T> bp{};
        for (int j = 0; j <= L; ++j) {
            bp.r[j] = V[j];
            bp.u[j] = U[j];
        }
        gstride = 4 * (L + 1);
        DS_CHECK(n4.alloc(4));
        DS_CHECK(da.alloc(4));
        DS_CHECK(db.alloc(4));
        DS_CHECK(gram.alloc((size_t)gstride * (L + 1)));
        DS_CHECK(coef.alloc(2 + MAXL));
        DS_CHECK(scal.alloc(1));
        dstate* S = dst.p;
        const int* skip = reliable ? &S->stop : &S->done;
        const unsigned vg = vgrid(h, n);
        T* part = reinterpret_cast<T*>(h->part);
        const bool recalc = !reliable && prm.resid_recalc_freq == 1;
        HPB_HIP(hipStreamSynchronize(st));
        HPB_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
        int rc = [&]() -> int {
            for (int j = 0; j < L; ++j) {
                hipLaunchKernelGGL((k_bs_upd_u<T>), dim3(vg), dim3(DB), 0, st, n, j, bp, coef.p, skip);
                ds_spmv<0, EPI_ALPHA>(U[j], nullptr, U[j + 1], rt, skip);
                hipLaunchKernelGGL((k_bs_upd_r<T>), dim3(vg), dim3(DB), 0, st, n, j, bp, P.x, coef.p, skip);
                if (j + 1 < L) ds_spmv<0, EPI_BETA>(V[j], nullptr, V[j + 1], rt, skip);
                else ds_spmv<0, EPI_NONE>(V[j], nullptr, V[j + 1], rt, skip);
            }
            switch (L) {
            case 1: ds_gram<1>(bp, skip); break;
            case 2: ds_gram<2>(bp, skip); break;
            case 3: ds_gram<3>(bp, skip); break;
            default: ds_gram<4>(bp, skip); break;
            }
            const int epi = reliable ? EPI_REL : EPI_CHECK;
            if (recalc) {
                if (comp)
                    hipLaunchKernelGGL((k_bs_upd_mr<T, true>), dim3(vg), dim3(DB), 0, st, n, L, bp, P.x, coef.p, skip);
                else
                    hipLaunchKernelGGL((k_bs_upd_mr<T, false>), dim3(vg), dim3(DB), 0, st, n, L, bp, P.x, coef.p, skip);
                ds_spmv<1, EPI_CHECK>(P.x, P.b, V[0], rt, skip);
            } else {
                const unsigned rg = rgrid(h, n);
                if (comp)
                    hipLaunchKernelGGL((k_ds_upd_mr<T, true>), dim3(rg), dim3(DB), 0, st, n, L, bp, P.x, rt, coef.p,
                                       part, skip);
                else
                    hipLaunchKernelGGL((k_ds_upd_mr<T, false>), dim3(rg), dim3(DB), 0, st, n, L, bp, P.x, rt,
                                       coef.p, part, skip);
                if (epi == EPI_REL) ds_fin<EPI_REL>(rg, skip);
                else ds_fin<EPI_CHECK>(rg, skip);
            }
            return HPB_OK;
        }();
        return end_capture<T>(st, gg, rc);
    }

    int run_bicgstabl(dstate* out)
    {
        hpb_handle_t h = P.h;
        hipStream_t st = h->stream;
        const size_t n = (size_t)P.rows;
        const int L = prm.basis;
        const bool comp = prm.high_precision != 0;
        const unsigned vg = vgrid(h, n);
        dstate* S = dst.p;
        // ||b||, tol, r_0 = b - A x, r~ = r_0 / ||r_0||, u_0 = 0
        DS_CHECK(nrm2_async<T>(h, n, P.b, n4.p, comp, nullptr));
        hipLaunchKernelGGL((k_init<T>), dim3(1), dim3(1), 0, st, S, n4.p, prm.rel_tol, prm.abs_tol);
        DS_CHECK(apply(P.x, P.b, V[0], nullptr));
        DS_CHECK(nrm2_async<T>(h, n, V[0], n4.p, comp, nullptr));
        hipLaunchKernelGGL((k_bs_init<T>), dim3(1), dim3(1), 0, st, S, n4.p, scal.p, hist());
        hipLaunchKernelGGL((k_scale_copy<T>), dim3(vg), dim3(DB), 0, st, n, V[0], rt, scal.p, &S->invalid);
        hipLaunchKernelGGL((k_fill<T>), dim3(vg), dim3(DB), 0, st, n, U[0], T(0));
        HPB_LAUNCH_CHECK();
        DS_CHECK(fused_beta(&S->done));
        DS_CHECK(read_state<T>(h, S, out));
        if (out->done) return HPB_OK;
        const int max_cycles = prm.max_iters / L + 2;
        const int every = 4;
        for (int c = 0; c < max_cycles; c += every) {
            for (int k = 0; k < every; ++k) HPB_HIP(hipGraphLaunch(gg.e, st));
            DS_CHECK(read_state<T>(h, S, out));
            if (out->done) break;
        }
        return HPB_OK;
    }

    // FP64 update: x64 += x32, x32 = 0, r64 = b64 - A64 x64 (compensated rows),
    // monitor check on ||r64||, r32 = (float) r64 (and on the first call r~, u_0)
    int rel_update(int first, int force_restart = 0)
    {
        hpb_handle_t h = P.h;
        hipStream_t st = h->stream;
        const size_t n = (size_t)P.rows;
        const unsigned vg = vgrid(h, n);
        dstate* S = dst.p;
        if (!first)
            hipLaunchKernelGGL(k_rel_flush, dim3(vg), dim3(DB), 0, st, n, (float*)P.x, R.x, S, &S->done);
        DS_CHECK(csr_apply<double>(h, P.rows, P.nnz, P.rp, P.ci, R.val, R.x, R.b, r64.p, true, &S->done));
        DS_CHECK(nrm2_async<double>(h, n, r64.p, n4d.p, true, &S->done));
        hipLaunchKernelGGL(k_rel_after, dim3(1), dim3(1), 0, st, S, n4d.p, hist(), first | force_restart, R.mscale);
        hipLaunchKernelGGL(k_rel_convert, dim3(vg), dim3(DB), 0, st, n, r64.p, (float*)V[0], (float*)rt,
                           (float*)U[0], S);
        HPB_LAUNCH_CHECK();
        return fused_beta(&S->done);
    }

    int run_reliable(dstate* out)
    {
        hpb_handle_t h = P.h;
        hipStream_t st = h->stream;
        const size_t n = (size_t)P.rows;
        const int L = prm.basis;
        dstate* S = dst.p;
        DS_CHECK(nrm2_async<double>(h, n, R.b, n4d.p, true, nullptr));
        hipLaunchKernelGGL((k_init<double>), dim3(1), dim3(1), 0, st, S, n4d.p, prm.rel_tol, prm.abs_tol);
        hipLaunchKernelGGL((k_fill<T>), dim3(vgrid(h, n)), dim3(DB), 0, st, n, P.x, T(0));
        DS_CHECK(rel_update(1));
        DS_CHECK(read_state<T>(h, S, out));
        const int max_cycles = prm.max_iters / L + 2;
        const int every = 4;
        constexpr int max_breakdown_restarts = 16;
        int cycles = 0, restarts = 0;
        while (cycles < max_cycles) {
            if (out->done) {
                // a breakdown restarts from an FP64 update; anything else ends the solve
                if (!out->breakdown || out->converged || out->invalid || out->iters >= prm.max_iters ||
                    restarts >= max_breakdown_restarts)
                    break;
                hipLaunchKernelGGL(k_rel_resume, dim3(1), dim3(1), 0, st, S);
                DS_CHECK(rel_update(0, 1));
                DS_CHECK(read_state<T>(h, S, out));
                restarts++;
                updates++;
                continue;
            }
            for (int k = 0; k < every; ++k) HPB_HIP(hipGraphLaunch(gg.e, st));
            cycles += every;
            DS_CHECK(read_state<T>(h, S, out));
            if (!out->done && out->stop) {
                DS_CHECK(rel_update(0));
                DS_CHECK(read_state<T>(h, S, out));
                updates++;
            }
        }
        // keep the progress of an unfinished run (x32 holds the increment since the last update)
        hipLaunchKernelGGL(k_rel_flush, dim3(vgrid(h, n)), dim3(DB), 0, st, n, (float*)P.x, R.x, S, &S->invalid);
        HPB_LAUNCH_CHECK();
        return HPB_OK;
    }

public:
    // one product as a solve forms it; *diagonals: K of the sliced form, 0 for CSR
    int product(const problem<T>& pr, const hpb_solver_params& p, const T* x, const T* b, T* y, int* diagonals)
    {
        P = pr;
        prm = p;
        target = p.rel_tol;
        DS_CHECK(plan_sdia());
        DS_CHECK(alloc_vectors(0, 0, 0));
        if (diagonals) *diagonals = A.K;
        if (y) DS_CHECK(apply(x, b, y, nullptr));
        HPB_HIP(hipStreamSynchronize(P.h->stream));
        return HPB_OK;
    }

    int updates = 0;
    bool fused = false;   // BiCGStab(L): the cycle graph finishes with beta for the next cycle

    // fused cycle: beta and rho for the first BiCG step from the current r_0
    int fused_beta(const int* skip)
    {
        if (!fused) return HPB_OK;
        hpb_handle_t h = P.h;
        DS_CHECK(dot2_async<T>(h, (size_t)P.rows, V[0], rt, da.p, prm.high_precision != 0, skip));
        hipLaunchKernelGGL((k_bs_beta<T>), dim3(1), dim3(1), 0, h->stream, dst.p, da.p, coef.p, 1, skip);
        HPB_LAUNCH_CHECK();
        return HPB_OK;
    }
};

}  // namespace

// Device-resident solve of A x = b (vectors of type T, scalars FP64).  Fills res
// (iters, converged, breakdown, resid_norm, rhs_norm, history_len) and history.
// cache (optional): a solver object kept by the caller between calls with the
// same operands; *cache is replaced when the operands or parameters change and
// must be released with dsolve_release.  target_tol: with a cache, the relative tolerance
// the solves reach together.
template <typename T>
int dsolve(hpb_handle_t h, int rows, int64_t nnz, const int* rp, const int* ci, const T* val, const T* b, T* x,
           const hpb_solver_params& p, hpb_solver_result* res, double* history, int history_cap,
           dsolver_base** cache, double target_tol)
{
    HPB_REQUIRE(p.solver != HPB_SOLVER_GMRES || (p.restart >= 1 && p.restart < MAXB), HPB_ERR_INVALID,
                "device solver: GMRES restart must be in [1, 255]");
    HPB_REQUIRE(p.solver != HPB_SOLVER_BICGSTABL || (p.basis >= 1 && p.basis <= MAXL), HPB_ERR_UNSUPPORTED,
                "device solver: BiCGStab(L) needs 1 <= L <= 8");
    const int hcap = (history && history_cap > 0) ? history_cap : 0;
    problem<T> P{h, rows, nnz, rp, ci, val, b, x};
    dsolver<T>* ds = nullptr;
    dsolver<T> local;
    if (cache && *cache) {
        ds = static_cast<dsolver<T>*>(*cache);
        if (!ds->matches(P, p, hcap)) {
            delete ds;
            *cache = nullptr;
            ds = nullptr;
        }
    }
    if (!ds) {
        ds = cache ? new dsolver<T>() : &local;
        const int rc = ds->setup(P, p, hcap, cache ? target_tol : p.rel_tol);
        if (rc != HPB_OK) {
            if (cache) delete ds;
            return rc;
        }
        if (cache) *cache = ds;
    }
    dstate out{};
    DS_CHECK(ds->run(p, &out));
    res->iters = out.iters;
    res->converged = out.converged;
    res->breakdown = out.breakdown;
    res->resid_norm = out.rnorm;
    res->rhs_norm = out.bnorm;
    res->history_len = out.hist_len;
    if (hcap && out.hist_len > 0) {
        HPB_HIP(hipMemcpyAsync(history, ds->history(), sizeof(double) * 2 * (size_t)out.hist_len,
                               hipMemcpyDeviceToHost, h->stream));
        HPB_HIP(hipStreamSynchronize(h->stream));
    }
    return HPB_OK;
}

void dsolve_release(dsolver_base* cache) { delete cache; }

// FP32 BiCGStab(L) with reliable updates of an FP64 solution: val32 / val64 share
// rp / ci; b64, x64 FP64; r32, x32 FP32 work vectors of the caller.  The inner
// rel_tol is the reduction delta of the FP32 recursive residual that triggers an
// FP64 update; rel_tol is the final tolerance on ||b - A x|| / ||b||.
int dsolve_reliable(hpb_handle_t h, int rows, int64_t nnz, const int* rp, const int* ci, const float* val32,
                    double mscale, const double* val64, const double* b64, double* x64, float* r32, float* x32,
                    const hpb_solver_params& inner, double rel_tol, hpb_solver_result* res, int* updates)
{
    HPB_REQUIRE(inner.solver == HPB_SOLVER_BICGSTABL && inner.basis >= 1 && inner.basis <= MAXL, HPB_ERR_UNSUPPORTED,
                "reliable updates: BiCGStab(L <= 8) inner solver only");
    HPB_REQUIRE(inner.rel_tol > 0.0 && inner.rel_tol < 1.0, HPB_ERR_INVALID,
                "reliable updates: the inner rel_tol (update threshold) must be in (0, 1)");
    problem<float> P{h, rows, nnz, rp, ci, val32, r32, x32};
    hpb_solver_params p = inner;
    const double delta = p.rel_tol;
    p.rel_tol = rel_tol;   // the monitor tests the FP64 true residual against the final tolerance
    rel64 R{val64, b64, x64, delta, mscale};
    dsolver<float> ds;
    DS_CHECK(ds.setup(P, p, 0, rel_tol, &R));
    dstate out{};
    DS_CHECK(ds.run(p, &out));
    res->iters = out.iters;
    res->converged = out.converged;
    res->breakdown = out.breakdown;
    res->resid_norm = out.rlast;
    res->rhs_norm = out.bnorm;
    res->history_len = 0;
    if (updates) *updates = ds.updates;
    return HPB_OK;
}

// 2^-e with max |x_i| 2^-e in [0.5, 1): scaling FP64 values by it before the
// conversion to FP32 changes no significand, and keeps |a_ij| < 1 in the FP32 copy
int absmax_pow2_scale(hpb_handle_t h, size_t n, const double* x, double* scale)
{
    HPB_REQUIRE(h && scale && (n == 0 || x), HPB_ERR_INVALID, "absmax: null argument");
    *scale = 1.0;
    if (n == 0) return HPB_OK;
    auto* d = reinterpret_cast<unsigned long long*>(h->dres);
    HPB_HIP(hipMemsetAsync(d, 0, sizeof(unsigned long long), h->stream));
    hipLaunchKernelGGL(k_absmax, dim3(vgrid(h, n)), dim3(DB), 0, h->stream, n, x, d);
    HPB_LAUNCH_CHECK();
    HPB_HIP(hipMemcpyAsync(h->hres, d, sizeof(unsigned long long), hipMemcpyDeviceToHost, h->stream));
    HPB_HIP(hipStreamSynchronize(h->stream));
    double m;
    std::memcpy(&m, h->hres, sizeof m);
    if (m > 0.0 && std::isfinite(m)) *scale = std::ldexp(1.0, -(std::ilogb(m) + 1));
    return HPB_OK;
}

template int dsolve<double>(hpb_handle_t, int, int64_t, const int*, const int*, const double*, const double*,
                            double*, const hpb_solver_params&, hpb_solver_result*, double*, int, dsolver_base**, double);
template int dsolve<float>(hpb_handle_t, int, int64_t, const int*, const int*, const float*, const float*, float*,
                           const hpb_solver_params&, hpb_solver_result*, double*, int, dsolver_base**, double);

}  // namespace hpb

namespace {
template <typename T>
int product_entry(hpb_handle_t h, int rows, int64_t nnz, const int* rp, const int* ci, const T* val,
                  const hpb_solver_params* p, const T* x, const T* b, T* y, int* diagonals)
{
    HPB_CLEAR_STALE();
    HPB_REQUIRE(h && rp && ci && val && p && (!y || x), HPB_ERR_INVALID, "hpb_csr_solver_product: null argument");
    HPB_REQUIRE(rows > 0 && nnz > 0, HPB_ERR_INVALID, "hpb_csr_solver_product: empty matrix");
    hpb::dsolver<T> ds;
    return ds.product(hpb::problem<T>{h, rows, nnz, rp, ci, val, nullptr, nullptr}, *p, x, b, y, diagonals);
}
}  // namespace

extern "C" {

int hpb_csr_solver_product_f64(hpb_handle_t h, int rows, int64_t nnz, const int* row_ptr, const int* col_ind,
                               const double* val, const hpb_solver_params* p, const double* x, const double* b,
                               double* y, int* diagonals)
{
    return product_entry<double>(h, rows, nnz, row_ptr, col_ind, val, p, x, b, y, diagonals);
}
int hpb_csr_solver_product_f32(hpb_handle_t h, int rows, int64_t nnz, const int* row_ptr, const int* col_ind,
                               const float* val, const hpb_solver_params* p, const float* x, const float* b, float* y,
                               int* diagonals)
{
    return product_entry<float>(h, rows, nnz, row_ptr, col_ind, val, p, x, b, y, diagonals);
}

}  // extern "C"
