// hpb_trsv.hip -- sparse triangular solves and ILU(0) for CSR matrices.
//
// Replaces csr::gpu_matrix::triangular_solve_lower / _upper
// (source/common/csr/gpu_matrix.h:142-320), which run cuSPARSE csrsv2 with a
// buffer-size query, an analysis, a cudaMalloc and the solve on every call:
//   lower: L x = alpha b with the strictly lower triangle and a unit diagonal
//          (CUSPARSE_DIAG_TYPE_UNIT: the stored diagonal is ignored);
//   upper: U x = alpha b with the upper triangle including the stored diagonal.
// The transposed solves of the reference (L^T x = alpha b, U^T x = alpha b) are the
// upper solve with a unit diagonal and the lower solve with the stored diagonal on
// the transpose of the matrix (hpb_csr_transpose_*); the analysis therefore also
// takes those two kinds (uplo 2: lower, stored diagonal; 3: upper, unit diagonal).
// Both read only their triangle, so one CSR holding an incomplete LU factorisation
// (L strictly below, U on and above the diagonal) serves both solves, as in the
// reference's csr::preconditioner (common/csr/preconditioner.h:61-75).
//
// Design: the analysis is done once per pattern and kept in an hpb_trsv_t: the
// level of every row (longest dependency chain, a host pass over row_ptr/col_ind
// in dependency order), the rows grouped by level, and the diagonal positions.
// Patterns of many narrow levels are solved in one launch whose rows wait for the
// values they need (k_trsv_flow, one lane per row); the others launch one kernel per
// level (k_trsv), the rows of a level being independent: LPR lanes per row (as in the
// SpMV) accumulate alpha b_i - sum a_ij x_j, merged by an xor butterfly.  Both are
// plain (fma) or compensated (Dot2 over the row).
// x may alias b: each row reads its own b_i before writing x_i.
//
// ILU(0) (new: the reference's gpu_ilu0_preconditioner::apply only copies its
// argument, common/csr/gpu_ilu0_preconditioner.h:62-72): the factors keep the
// pattern of A and satisfy (L U)_ij = a_ij on it.  Row i is finished level by level
// with the lower analysis (it depends on the rows k < i it references): for
// k in row i in increasing order, l_ik = a_ik / u_kk, then a_ij -= l_ik u_kj for
// every j > k present in both rows; one 64-lane block per row, lanes over j.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <thread>
#include <type_traits>
#include <vector>

#include "hpb_device.hpp"
#include "hpb_internal.hpp"

struct hpb_trsv_s {
    int uplo = 0;        // 0 lower (unit diagonal), 1 upper, 2 lower (stored diagonal), 3 upper (unit diagonal)
    bool upper = false;
    bool unit = true;
    int rows = 0;
    int64_t nnz = 0;
    const int* rp = nullptr;    // the caller's device arrays (not owned)
    const int* ci = nullptr;
    int* perm = nullptr;        // device: rows ordered by level
    int* diag = nullptr;        // device: position of the diagonal entry of each row, -1 if absent
    std::vector<int> level_ptr; // host: level l holds perm[level_ptr[l] .. level_ptr[l+1])
    int lpr = 1;
    bool all_diag = false;      // every row stores its diagonal entry
    int4* recs = nullptr;       // device, rows by level: {row, first dependency, their number | 256 x the lane of the
                                // first in the level kernels, diagonal entry}; null: the level kernels solve this pattern
};

namespace hpb {
namespace {

constexpr int TB = 256;

template <typename T, int LPR, bool COMP, bool UPPER, bool UNIT>
__global__ __launch_bounds__(TB) void k_trsv(int beg, int end, const int* __restrict__ perm,
                                             const int* __restrict__ rp, const int* __restrict__ ci,
                                             const T* __restrict__ val, const int* __restrict__ diag, T alpha,
                                             const T* b, T* x)
{
    const int lane = threadIdx.x % LPR;
    const int t = beg + (int)((blockIdx.x * TB + threadIdx.x) / LPR);
    if (t >= end) return;
    const int i = perm[t];
    const int rb = rp[i], re = rp[i + 1];
    T s = T(0), c = T(0);
    if (lane == 0) s = alpha == T(1) ? b[i] : alpha * b[i];
    for (int k = rb + lane; k < re; k += LPR) {
        const int j = ci[k];
        if (UPPER ? (j > i) : (j < i)) {
            if (COMP) dev::dot2_step<T>(s, c, -val[k], x[j]);
            else s = dev::fma_rn<T>(-val[k], x[j], s);
        }
    }
#pragma unroll
    for (int m = LPR / 2; m >= 1; m >>= 1) {
        const T s2 = __shfl_xor(s, m, 64);
        if (COMP) {
            const T c2 = __shfl_xor(c, m, 64);
            dev::merge<T>(s, c, s2, c2);
        } else {
            s = s + s2;
        }
    }
    if (lane == 0) {
        T v = COMP ? s + c : s;
        if (!UNIT) v = v / val[diag[i]];
        x[i] = v;
    }
}

// ---- one launch for all levels
//
// Patterns with many narrow levels are bound by the latency of a launch per level (3.6 us
// each).  Here waves take chunks of 64 rows in level order, one row per lane, from a
// counter, and each row waits for the values it depends on: the solution is also kept in
// `w`, which starts as the bit pattern FLOW_EMPTY, and a lane polls the entries of w it
// needs (relaxed agent-scope loads: value and readiness in one 8- or 4-byte word).  Rows
// only depend on earlier levels, so on earlier positions of the chunk order: the wave
// that holds the smallest unfinished chunk never waits for a chunk nobody has taken, and
// every wait ends whatever waves are resident; a row of the same wave is stored inside
// the polling loop, whose exit is uniform.  (The polls are bounded all the same: after
// hpb_handle_s::flow_spins polls for its chunk a wave takes NaN for the values that are
// missing and marks the handle's host record, which its next call that waits reports.  The
// longest legal wait, 256 chunks of 64 levels in turn, is some 20 ms, the bound seconds.)
// About four levels' rows are in
// flight, so that a wave has its entries loaded when its level comes up; more pollers
// slow the chain.
// A plain row is summed as the LPR lanes of the level kernel sum it, entries LPR apart in
// one sum each and the sums added in pairs, so its bits are the level kernel's: one serial
// sum of 40 entries has 2.4 times the rounding error.  The four sums the next entries go
// to stay in acc[0 .. 3]: acc turns by four after every four entries, and the pairs it is
// added in are the same however far it has turned.  (One serial sum instead: 7-point
// 128^3 681 us against 684, 150 levels of 300 rows of 24 entries 214 against 222.)  A
// compensated row is one Dot2 sum.
// 96 x 90 x 84 7-point (268 levels), lower / upper: 421 / 422 us, with a launch per level
// 967 / 1083; 5-point 1000^2 (1999 levels) 2348 / 2404 (7191 / 8126); tridiagonal, 20 000
// levels of one row, 13.4 / 14.0 ms (76.5 / 70.8).
template <typename T> struct flow_bits;
template <> struct flow_bits<double> {
    using type = unsigned long long;
    static constexpr type empty = 0xfff8a5c30f1e2d4bull, nan = 0x7ff8000000000000ull;
};
template <> struct flow_bits<float> {
    using type = unsigned;
    static constexpr type empty = 0xffc5a30fu, nan = 0x7fc00000u;
};

// w := FLOW_EMPTY, *next := 0
template <typename T>
__global__ __launch_bounds__(TB) void k_flow_init(int rows, typename flow_bits<T>::type* __restrict__ w,
                                                  unsigned* __restrict__ next)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) *next = 0u;
    for (long i = (long)blockIdx.x * TB + threadIdx.x; i < rows; i += (long)gridDim.x * TB) w[i] = flow_bits<T>::empty;
}

template <typename T, bool COMP, bool UNIT, int LPR>
__global__ __launch_bounds__(64) void k_trsv_flow(int rows, const int4* __restrict__ recs, const int* __restrict__ ci,
                                                  const T* __restrict__ val, T alpha, const T* b, T* x,
                                                  typename flow_bits<T>::type* w, unsigned* next, unsigned spins,
                                                  int* gave_up)
{
    using U = typename flow_bits<T>::type;
    constexpr int NA = COMP ? 1 : LPR;
    const int lane = threadIdx.x;
    for (;;) {
        unsigned chunk = 0;
        if (lane == 0) chunk = __hip_atomic_fetch_add(next, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        chunk = __builtin_amdgcn_readfirstlane(chunk);
        const long t = (long)chunk * 64 + lane;
        if ((long)chunk * 64 >= rows) return;
        bool stored = t >= rows;
        const int4 rec = recs[stored ? rows - 1 : t];
        const int i = rec.x, end = rec.y + (rec.z & 255);
        int p = rec.y;
        const T bi = alpha == T(1) ? b[i] : alpha * b[i];
        const T d = UNIT ? T(1) : val[rec.w];
        T acc[NA], c = T(0);
        {
            const int at = -(rec.z >> 8) & (NA - 1);   // lane 0's sum starts from b_i
#pragma unroll
            for (int k = 0; k < NA; ++k) acc[k] = k == at ? bi : T(0);
        }
        // four entries at a time: columns, values and (once there) the solution values
        int j[4];
        T a[4], xv[4];
        unsigned wait = 0;   // entries whose solution value is not there yet
        auto fetch = [&]() {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const bool has = p + q < end;
                j[q] = has ? ci[p + q] : i;
                a[q] = has ? val[p + q] : T(0);
                xv[q] = T(0);
                if (has) wait |= 1u << q;
            }
        };
        if (!stored) fetch();
        // spin: uniform, and never reset (counts per lane or since the last row cost 1 to 2 %)
        for (unsigned spin = 0; __ballot(!stored) != 0; ++spin) {
            if (stored) continue;
            U v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = __hip_atomic_load(w + j[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (((wait >> q) & 1u) && (v[q] != flow_bits<T>::empty || spin >= spins)) {
                    xv[q] = __builtin_bit_cast(T, v[q]);
                    wait &= ~(1u << q);
                }
            if (wait == 0) {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (p + q < end) {
                        if (COMP) dev::dot2_step<T>(acc[0], c, -a[q], xv[q]);
                        else acc[q % NA] = dev::fma_rn<T>(-a[q], xv[q], acc[q % NA]);
                    }
                p += 4;
                if (p < end) {
                    fetch();
                    if constexpr (NA > 4) {
                        T turned[NA];
#pragma unroll
                        for (int k = 0; k < NA; ++k) turned[k] = acc[(k + 4) % NA];
#pragma unroll
                        for (int k = 0; k < NA; ++k) acc[k] = turned[k];
                    }
                } else {
#pragma unroll
                    for (int m = NA / 2; m >= 1; m >>= 1)
#pragma unroll
                        for (int k = 0; k < NA / 2; ++k)
                            if (k < m) acc[k] = acc[k] + acc[k + m];
                    T r = COMP ? acc[0] + c : acc[0];
                    if (!UNIT) r = r / d;
                    U bits = __builtin_bit_cast(U, r);
                    if (bits == flow_bits<T>::empty) bits = flow_bits<T>::nan;   // this NaN means "not there"
                    __hip_atomic_store(w + i, bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    x[i] = r;
                    if (spin >= spins) __hip_atomic_store(gave_up, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                    stored = true;
                }
            }
        }
    }
}

// hpb_trsv_s::recs
__global__ __launch_bounds__(TB) void k_flow_recs(int rows, bool upper, int lpr, const int* __restrict__ perm,
                                                  const int* __restrict__ rp, const int* __restrict__ ci,
                                                  const int* __restrict__ diag, int4* __restrict__ recs)
{
    for (long t = (long)blockIdx.x * TB + threadIdx.x; t < rows; t += (long)gridDim.x * TB) {
        const int i = perm[t], rb = rp[i], re = rp[i + 1];
        int lo = rb, hi = re;   // first entry with column >= i (columns are sorted)
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (ci[mid] < i) lo = mid + 1;
            else hi = mid;
        }
        const int d = diag[i], after = lo + (d >= 0 ? 1 : 0);
        recs[t] = upper ? make_int4(i, after, (re - after) | (after - rb) % lpr << 8, d) : make_int4(i, rb, lo - rb, d);
    }
}

template <typename T>
__global__ __launch_bounds__(64) void k_ilu0_rows(int beg, const int* __restrict__ perm, const int* __restrict__ rp,
                                                  const int* __restrict__ ci, const int* __restrict__ diag,
                                                  T* __restrict__ val)
{
    const int i = perm[beg + blockIdx.x];
    const int rb = rp[i], re = rp[i + 1], di = diag[i];
    for (int kk = rb; kk < di; ++kk) {
        const int k = ci[kk];
        const T lik = val[kk] / val[diag[k]];
        __syncthreads();   // every lane has read val[kk] before it changes
        if (threadIdx.x == 0) val[kk] = lik;
        // a_ij -= l_ik u_kj for j > k in row i that also appear in row k (upper part)
        const int kb = diag[k] + 1, ke = rp[k + 1];
        for (int jj = kk + 1 + (int)threadIdx.x; jj < re; jj += 64) {
            const int j = ci[jj];
            int lo = kb, hi = ke;   // binary search of column j in row k's upper part
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (ci[mid] < j) lo = mid + 1;
                else hi = mid;
            }
            if (lo < ke && ci[lo] == j) val[jj] = dev::fma_rn<T>(-lik, val[lo], val[jj]);
        }
        __syncthreads();   // row i updated before the next k reads it
    }
}

template <typename T, bool COMP, bool UPPER, bool UNIT, int LPR>
void trsv_level(hipStream_t st, const hpb_trsv_s* t, int beg, int end, const T* val, T alpha, const T* b, T* x)
{
    const int rows = end - beg;
    const int per_block = TB / LPR;
    const unsigned grid = (unsigned)((rows + per_block - 1) / per_block);
    hipLaunchKernelGGL((k_trsv<T, LPR, COMP, UPPER, UNIT>), dim3(grid), dim3(TB), 0, st, beg, end, t->perm, t->rp,
                       t->ci, val, t->diag, alpha, b, x);
}

// Waves of a one-launch solve: the rows of four levels of average width, at most one wave
// per CU.  Lower solve, us, at 1 / 2 / 4 / 8 / 16 levels' rows: 7-point 96 x 90 x 84 (2.7 k
// rows per level) 602 / 414 / 421 / 505 / 686, 128^3 (5.5 k) 863 / 646 / 749 / 1018 / 1297,
// 5-point 1000^2 (0.5 k) 3755 / 2477 / 2348 / 2465 / 2593, random rows 300 k x 20 (5.4 k)
// 304 / 168 / 121 / 137 / 181: fewer leave a level without its entries loaded, more slow
// the chain by polling.
long flow_waves(int rows, int nlev, long cus)
{
    const long width = ((long)rows + nlev - 1) / nlev;
    return std::max(8L, std::min(cus, (4 * width + 63) / 64));
}

// Whether one launch for all levels beats a launch per level.  It saves about 2 us a level,
// but one lane walks each row, 64 rows to a wave, and the waves at work are few: long rows
// cost a start of their own, wide levels fill the device better in a launch each.  Lower
// solves of levels of equal width, plain, one launch / a launch per level, us:
//   2 dependencies: 4 levels of 100 rows 8 / 11, of 6000 14 / 12; 12 of 6000 25 / 33;
//     150 of 15 000 436 / 557, of 22 000 632 / 563;
//   12: 6 levels of 1000 16 / 18, of 6000 23 / 18; 50 of 11 000 150 / 178, of 15 000 197 / 196;
//   24: 14 levels of 300 35 / 40, of 3000 45 / 42; 26 of 3000 64 / 89; 50 of 11 000 220 / 227;
//   48: 26 levels of 300 78 / 79 (compensated 89 / 84); 50 of 300 134 / 154, of 8000 280 / 268;
//   60: 12 levels of 1000 56 / 40, 40 of 1000 137 / 178.
// 7-point grids, 256^3 (766 levels, 21.9 k rows on average) 3507 / 4278; 100 000 random rows
// of 2.6 dependencies, the longest of 20, in 26 levels 39 / 85.
bool flow_pays(int rows, int nlev, int longest, int64_t deps)
{
    const double width = (double)rows / nlev, per_level = (double)deps / nlev;
    const double length = std::max((double)deps / rows, 0.5 * longest);
    if (longest > 64 || per_level > 250000.0) return false;
    if (width <= 1024.0) return nlev >= std::max(4.0, 0.6 * length);
    if (width > (nlev < 24 ? 8192.0 : nlev < 100 ? 11264.0 : nlev < 500 ? 16384.0 : 24576.0)) return false;
    return nlev >= (length <= 4.0 ? 6.0 : std::max(12.0, 0.75 * length));
}

// The handle's workspace of one-launch solves, at least `bytes`; null when it cannot be
// had (no memory, or the stream is being captured and it would have to grow).  A buffer
// that is outgrown stays allocated until the handle goes: a captured solve may use it.
char* flow_workspace(hpb_handle_t h, size_t bytes)
{
    if (h->flow_bytes >= bytes) return static_cast<char*>(h->flow.back());
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(h->stream, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone) {
        (void)hipGetLastError();
        return nullptr;
    }
    const size_t want = std::max(bytes, 2 * h->flow_bytes);
    void* p = nullptr;
    if (hipMalloc(&p, want) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    h->flow.push_back(p);
    h->flow_bytes = want;
    return static_cast<char*>(p);
}
size_t flow_bytes_of(int rows) { return 64 + sizeof(double) * (size_t)rows; }

template <typename T, bool COMP, bool UPPER, bool UNIT>
void trsv_all(hpb_handle_t h, const hpb_trsv_s* t, const T* val, T alpha, const T* b, T* x)
{
    hipStream_t st = h->stream;
    const int nl = (int)t->level_ptr.size() - 1;
    char* ws = t->recs ? flow_workspace(h, flow_bytes_of(t->rows)) : nullptr;
    if (ws) {
        using U = typename flow_bits<T>::type;
        U* w = reinterpret_cast<U*>(ws + 64);
        unsigned* next = reinterpret_cast<unsigned*>(ws);
        const long cus = h->num_cu > 0 ? h->num_cu : 256;
        const unsigned gi = (unsigned)std::max(1L, std::min(((long)t->rows + TB - 1) / TB, 4 * cus));
        hipLaunchKernelGGL((k_flow_init<T>), dim3(gi), dim3(TB), 0, st, t->rows, w, next);
        auto go = [&](auto lprc) {
            hipLaunchKernelGGL((k_trsv_flow<T, COMP, UNIT, decltype(lprc)::value>),
                               dim3((unsigned)flow_waves(t->rows, nl, cus)), dim3(64), 0, st, t->rows, t->recs, t->ci,
                               val, alpha, b, x, w, next, h->flow_spins, &host_flag_of(h)->flow_gave_up);
        };
        if (COMP || t->lpr == 1) go(std::integral_constant<int, 1>{});
        else if (t->lpr == 2) go(std::integral_constant<int, 2>{});
        else if (t->lpr == 4) go(std::integral_constant<int, 4>{});
        else if (t->lpr == 8) go(std::integral_constant<int, 8>{});
        else go(std::integral_constant<int, 16>{});
        return;
    }
    for (int l = 0; l < nl; ++l) {
        const int beg = t->level_ptr[l], end = t->level_ptr[l + 1];
        switch (t->lpr) {
        case 1: trsv_level<T, COMP, UPPER, UNIT, 1>(st, t, beg, end, val, alpha, b, x); break;
        case 2: trsv_level<T, COMP, UPPER, UNIT, 2>(st, t, beg, end, val, alpha, b, x); break;
        case 4: trsv_level<T, COMP, UPPER, UNIT, 4>(st, t, beg, end, val, alpha, b, x); break;
        case 8: trsv_level<T, COMP, UPPER, UNIT, 8>(st, t, beg, end, val, alpha, b, x); break;
        default: trsv_level<T, COMP, UPPER, UNIT, 16>(st, t, beg, end, val, alpha, b, x); break;
        }
    }
}

template <typename T>
int trsv_entry(hpb_handle_t h, hpb_trsv_t t, const T* val, T alpha, const T* b, T* x, int comp)
{
    HPB_CLEAR_STALE();
    HPB_REQUIRE(h && t && val && b && x, HPB_ERR_INVALID, "hpb_csr_trsv: null argument");
    if (const int rc = flow_status(h)) return rc;   // an earlier solve's
    switch (t->uplo) {
    case 0:
        if (comp) trsv_all<T, true, false, true>(h, t, val, alpha, b, x);
        else trsv_all<T, false, false, true>(h, t, val, alpha, b, x);
        break;
    case 1:
        if (comp) trsv_all<T, true, true, false>(h, t, val, alpha, b, x);
        else trsv_all<T, false, true, false>(h, t, val, alpha, b, x);
        break;
    case 2:
        if (comp) trsv_all<T, true, false, false>(h, t, val, alpha, b, x);
        else trsv_all<T, false, false, false>(h, t, val, alpha, b, x);
        break;
    default:
        if (comp) trsv_all<T, true, true, true>(h, t, val, alpha, b, x);
        else trsv_all<T, false, true, true>(h, t, val, alpha, b, x);
        break;
    }
    HPB_LAUNCH_CHECK();
    return HPB_OK;
}

template <typename T>
int ilu0_entry(hpb_handle_t h, hpb_trsv_t t, T* val)
{
    HPB_CLEAR_STALE();
    HPB_REQUIRE(h && t && val, HPB_ERR_INVALID, "hpb_csr_ilu0: null argument");
    HPB_REQUIRE(t->uplo == 0, HPB_ERR_INVALID, "hpb_csr_ilu0: needs the analysis of the lower triangle");
    HPB_REQUIRE(t->all_diag, HPB_ERR_INVALID, "hpb_csr_ilu0: every row needs a stored diagonal entry");
    const int nl = (int)t->level_ptr.size() - 1;
    for (int l = 0; l < nl; ++l) {
        const int beg = t->level_ptr[l], end = t->level_ptr[l + 1];
        hipLaunchKernelGGL((k_ilu0_rows<T>), dim3((unsigned)(end - beg)), dim3(64), 0, h->stream, beg, t->perm, t->rp,
                           t->ci, t->diag, val);
    }
    HPB_LAUNCH_CHECK();
    return HPB_OK;
}

}  // namespace
}  // namespace hpb

using namespace hpb;

extern "C" {

int hpb_csr_trsv_analysis(hpb_handle_t h, int uplo, int rows, int64_t nnz, const int* row_ptr, const int* col_ind,
                          hpb_trsv_t* out)
{
    HPB_CLEAR_STALE();
    HPB_REQUIRE(h && row_ptr && col_ind && out, HPB_ERR_INVALID, "hpb_csr_trsv_analysis: null argument");
    HPB_REQUIRE(uplo >= 0 && uplo <= 3, HPB_ERR_INVALID, "hpb_csr_trsv_analysis: uplo must be 0, 1, 2 or 3");
    const bool lower = (uplo == 0 || uplo == 2), unit = (uplo == 0 || uplo == 3);
    HPB_REQUIRE(rows > 0 && nnz > 0 && nnz < (1ll << 31), HPB_ERR_INVALID, "hpb_csr_trsv_analysis: bad size");
    *out = nullptr;
    // the pattern on the host, through the handle's pinned staging buffer (a pageable
    // copy of the 128^3 pattern took 15-18 ms)
    const size_t need = sizeof(int) * ((size_t)rows + 1 + (size_t)nnz);
    if (h->hstage_bytes < need) {
        if (h->hstage) (void)hipHostFree(h->hstage);
        h->hstage = nullptr;
        h->hstage_bytes = 0;
        HPB_HIP(hipHostMalloc(&h->hstage, need, hipHostMallocDefault));
        h->hstage_bytes = need;
    }
    int* const rp = static_cast<int*>(h->hstage);
    int* const ci = rp + (size_t)rows + 1;
    HPB_HIP(hipMemcpyAsync(rp, row_ptr, sizeof(int) * ((size_t)rows + 1), hipMemcpyDeviceToHost, h->stream));
    HPB_HIP(hipMemcpyAsync(ci, col_ind, sizeof(int) * (size_t)nnz, hipMemcpyDeviceToHost, h->stream));
    HPB_HIP(hipStreamSynchronize(h->stream));
    HPB_REQUIRE(rp[0] == 0 && rp[rows] == nnz, HPB_ERR_INVALID, "hpb_csr_trsv_analysis: row_ptr inconsistent with nnz");
    // checks, diagonal positions and the end of each row's lower part (the columns
    // are sorted, so a row's j < i come first), in parallel over row ranges; the
    // first failing row in dependency order names the error, as a sequential scan
    std::vector<int> level((size_t)rows, 0), diag((size_t)rows, -1), lend((size_t)rows);
    {
        const unsigned hw = std::max(1u, std::thread::hardware_concurrency());
        const unsigned T = (unsigned)std::max<int64_t>(1, std::min<int64_t>({(int64_t)hw, 16, (int64_t)rows / 65536 + 1}));
        std::vector<int> first_code(T, 0);
        auto scan = [&](unsigned t) {
            const int s0 = (int)((int64_t)rows * t / T), s1 = (int)((int64_t)rows * (t + 1) / T);
            for (int s = s0; s < s1; ++s) {
                const int i = lower ? s : rows - 1 - s;   // dependency order
                int code = 0, le = rp[i + 1];
                for (int k = rp[i]; k < rp[i + 1]; ++k) {
                    const int j = ci[k];
                    if (!(j >= 0 && j < rows)) { code = 1; break; }
                    if (!(k == rp[i] || ci[k - 1] < j)) { code = 2; break; }
                    if (j >= i && le == rp[i + 1]) le = k;
                    if (j == i) diag[i] = k;
                }
                lend[i] = le;
                if (!code && !unit && diag[i] < 0) code = 3;
                if (code) {   // later rows of this range cannot come first
                    first_code[t] = code;
                    return;
                }
            }
        };
        std::vector<std::thread> th;
        for (unsigned t = 1; t < T; ++t) th.emplace_back(scan, t);
        scan(0);
        for (auto& x : th) x.join();
        for (unsigned t = 0; t < T; ++t) {   // ranges in dependency order: the first error wins
            HPB_REQUIRE(first_code[t] != 1, HPB_ERR_INVALID, "hpb_csr_trsv_analysis: column index out of range");
            HPB_REQUIRE(first_code[t] != 2, HPB_ERR_INVALID,
                        "hpb_csr_trsv_analysis: columns must be sorted and unique within a row");
            HPB_REQUIRE(first_code[t] != 3, HPB_ERR_INVALID,
                        "hpb_csr_trsv_analysis: a row without a stored diagonal entry (structurally singular)");
        }
    }
    // levels (longest dependency chain): one pass in dependency order over the
    // dependencies only
    int nlev = 0;
    for (int s = 0; s < rows; ++s) {
        const int i = lower ? s : rows - 1 - s;
        int lv = 0;
        if (lower) {
            for (int k = rp[i]; k < lend[i]; ++k) lv = std::max(lv, level[ci[k]] + 1);
        } else {
            for (int k = lend[i] + (diag[i] >= 0 ? 1 : 0); k < rp[i + 1]; ++k) lv = std::max(lv, level[ci[k]] + 1);
        }
        level[i] = lv;
        nlev = std::max(nlev, lv + 1);
    }
    hpb_trsv_s* t = new hpb_trsv_s();
    t->uplo = uplo;
    t->upper = !lower;
    t->unit = unit;
    t->rows = rows;
    t->nnz = nnz;
    t->rp = row_ptr;
    t->ci = col_ind;
    t->level_ptr.assign((size_t)nlev + 1, 0);
    for (int i = 0; i < rows; ++i) t->level_ptr[level[i] + 1]++;
    for (int l = 0; l < nlev; ++l) t->level_ptr[l + 1] += t->level_ptr[l];
    std::vector<int> perm((size_t)rows), fill(t->level_ptr.begin(), t->level_ptr.end() - 1);
    for (int i = 0; i < rows; ++i) perm[fill[level[i]]++] = i;   // ascending row order within a level
    t->all_diag = std::all_of(diag.begin(), diag.end(), [](int d) { return d >= 0; });
    const double mean = (double)nnz / rows;
    t->lpr = mean <= 1.5 ? 1 : mean <= 3.0 ? 2 : mean <= 6.0 ? 4 : mean <= 12.0 ? 8 : 16;
    int longest = 0;
    int64_t deps = 0;
    for (int i = 0; i < rows; ++i) {
        const int d = lower ? lend[i] - rp[i] : rp[i + 1] - lend[i];   // an upper row's diagonal counts
        longest = std::max(longest, d);
        deps += d;
    }
    const bool flow = flow_pays(rows, nlev, longest, deps);
    hipError_t e = hipMalloc((void**)&t->perm, sizeof(int) * rows);
    if (e == hipSuccess) e = hipMalloc((void**)&t->diag, sizeof(int) * rows);
    if (e == hipSuccess) e = hipMemcpyAsync(t->perm, perm.data(), sizeof(int) * rows, hipMemcpyHostToDevice, h->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(t->diag, diag.data(), sizeof(int) * rows, hipMemcpyHostToDevice, h->stream);
    if (e == hipSuccess && flow) {
        // without the memory for it the level kernels solve the pattern
        if (hipMalloc((void**)&t->recs, sizeof(int4) * rows) != hipSuccess) {
            t->recs = nullptr;
            (void)hipGetLastError();
        } else {
            const unsigned g = (unsigned)std::min(((long)rows + TB - 1) / TB, 4096L);
            hipLaunchKernelGGL(k_flow_recs, dim3(g), dim3(TB), 0, h->stream, rows, !lower, t->lpr, t->perm, t->rp, t->ci,
                               t->diag, t->recs);
            e = hipGetLastError();
            (void)flow_workspace(h, flow_bytes_of(rows));   // so that a captured solve finds it
        }
    }
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess) {
        if (t->perm) (void)hipFree(t->perm);
        if (t->diag) (void)hipFree(t->diag);
        if (t->recs) (void)hipFree(t->recs);
        delete t;
        return hip_status(e, __FILE__, __LINE__, "hpb_csr_trsv_analysis");
    }
    *out = t;
    return HPB_OK;
}

int hpb_csr_trsv_levels(hpb_trsv_t t, int* nlevels)
{
    HPB_REQUIRE(t && nlevels, HPB_ERR_INVALID, "hpb_csr_trsv_levels: null argument");
    *nlevels = (int)t->level_ptr.size() - 1;
    return HPB_OK;
}

int hpb_csr_trsv_launches(hpb_trsv_t t, int* launches)
{
    HPB_REQUIRE(t && launches, HPB_ERR_INVALID, "hpb_csr_trsv_launches: null argument");
    *launches = t->recs ? 2 : (int)t->level_ptr.size() - 1;
    return HPB_OK;
}

int hpb_trsv_destroy(hpb_trsv_t t)
{
    if (t) {
        if (t->perm) (void)hipFree(t->perm);
        if (t->diag) (void)hipFree(t->diag);
        if (t->recs) (void)hipFree(t->recs);
        delete t;
    }
    return HPB_OK;
}

int hpb_csr_trsv_f64(hpb_handle_t h, hpb_trsv_t t, const double* val, double alpha, const double* b, double* x,
                     int compensated)
{
    return trsv_entry<double>(h, t, val, alpha, b, x, compensated);
}
int hpb_csr_trsv_f32(hpb_handle_t h, hpb_trsv_t t, const float* val, float alpha, const float* b, float* x,
                     int compensated)
{
    return trsv_entry<float>(h, t, val, alpha, b, x, compensated);
}

int hpb_csr_ilu0_f64(hpb_handle_t h, hpb_trsv_t lower, double* val)
{
    return ilu0_entry<double>(h, lower, val);
}
int hpb_csr_ilu0_f32(hpb_handle_t h, hpb_trsv_t lower, float* val)
{
    return ilu0_entry<float>(h, lower, val);
}

}  // extern "C"
