// hpb_sdia.hpp -- sliced-diagonal form of a CSR matrix for repeated products.
//
// A solver multiplies by one matrix hundreds of times, so it first rewrites the CSR
// arrays (csr::matrix, source/common/csr/matrix.h:91-158) into slices of 64 rows, one
// row per lane of a wave.  A slice keeps K diagonals: the offset column - row, the same
// for the whole slice, a 64-bit mask of the rows that hold an entry on it, and 64 values
// stored lane by lane.  Against CSR a product then reads no column indices (4 of 12
// bytes of an FP64 entry, 4 of 8 of an FP32 one) and no row pointers, every load of
// values and of x is a contiguous run of the wave, and no LDS staging is needed.
// Grid operators in any row order that keeps runs of rows along a line fit (K = 5 or 7
// for the 5- and 7-point stencils, boundary rows are holes in the masks).  The form is
// taken when every row's columns are strictly ascending, no slice has more than
// SD_MAXK diagonals and the K 64-row columns of all slices hold at most a quarter more
// slots than the matrix has entries; any other matrix stays in CSR.
// Where the CSR kernels take two lanes per row (a mean of more than 1.5 and up to 8
// entries), a row's entries are summed as those lanes sum them (entries 0, 2, ... and 1,
// 3, ... apart, then merged): the bits are the same.  Longer plain rows keep as many sums
// as CSR has lanes, the diagonals dealt out in turn: the bits of CSR for rows that hold
// an entry on every diagonal of their slice, no longer chains for the others.  (Two sums
// instead: 1.1 to 1.3 times CSR's rounding error at 19 to 32 entries.)  Longer compensated
// rows stay with two Dot2 sums.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "hpb_device.hpp"

namespace hpb {

constexpr int SD_MAXK = 32;   // diagonals of a slice, at most
constexpr int SD_THREADS = 256;

template <typename T>
struct sdia_view {
    int K;                 // diagonals per slice (slices with fewer are padded with empty masks)
    const int* off;        // K per slice: column - row
    const uint64_t* mask;  // K per slice
    const T* val;          // 64 K per slice: lane by lane, zero where the mask is
};

namespace sd {

// Walks the diagonals of the slice of rows [r0, r1), at most 64, in ascending order, a
// wave per slice: f(k, offset, mask, position of this lane's entry or -1).  colat(p) is
// the column of entry p.  Returns the number of diagonals, or -1 when the slice does not
// fit (more than SD_MAXK, or columns not strictly ascending).
template <class C, class F>
__device__ __forceinline__ int walk_slice(long r0, long r1, const int* __restrict__ rp, C colat, F f)
{
    const int lane = threadIdx.x & 63;
    const long r = r0 + lane;
    int p = 0, e = 0;
    if (r < r1) {
        p = rp[r];
        e = rp[r + 1];
    }
    int prev = -1;   // the row's last column taken
    for (int k = 0;; ++k) {
        const int c = p < e ? colat(p) : 0;
        const int d = p < e ? (int)(c - r) : 2147483647;
        if (__ballot(p < e && c <= prev)) return -1;
        int m = d;
#pragma unroll
        for (int s = 32; s >= 1; s >>= 1) {
            const int o = __shfl_xor(m, s, 64);
            m = o < m ? o : m;
        }
        if (m == 2147483647) return k;
        if (k == SD_MAXK) return -1;
        const bool take = p < e && d == m;
        f(k, m, (uint64_t)__ballot(take), take ? p : -1);
        if (take) {
            prev = c;
            ++p;
        }
    }
}

// The wave's ne consecutive elements from src into its LDS area, eight loads in flight per
// lane: rows read by their lanes took a line per lane, step and array (1 M rows of 27
// entries: count 370 us, fill 890 us).
template <typename E>
__device__ __forceinline__ void wave_stage(const E* __restrict__ src, int ne, E* lds)
{
    const int lane = threadIdx.x & 63;
    for (int i = 0; i < ne; i += 512) {
        E t[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int at = i + q * 64 + lane;
            t[q] = src[at < ne ? at : ne - 1];
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int at = i + q * 64 + lane;
            if (at < ne) lds[at] = t[q];
        }
    }
}
// orders the LDS accesses of one wave across its lanes
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// info[0] = largest number of diagonals of a slice, info[1] != 0: some slice does not fit
__global__ __launch_bounds__(SD_THREADS) inline void k_sdia_count(long nsl, int rows, const int* __restrict__ rp,
                                                                  const int* __restrict__ col, int* __restrict__ info)
{
    constexpr int CAP = 64 * SD_MAXK;   // a slice that fits has no more entries
    __shared__ int lc[SD_THREADS / 64][CAP];
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long w = (long)blockIdx.x * (SD_THREADS / 64) + wid, nw = (long)gridDim.x * (SD_THREADS / 64);
    int most = 0;
    bool bad = false;
    for (long sl = w; sl < nsl && !bad; sl += nw) {
        const long r0 = sl * 64, r1 = r0 + 64 < rows ? r0 + 64 : rows;
        const int e0 = rp[r0], ne = rp[r1] - e0;
        if (ne > CAP) {
            bad = true;
            break;
        }
        wave_stage(col + e0, ne, lc[wid]);
        wave_sync();
        const int k = walk_slice(r0, r1, rp, [&](int p) { return lc[wid][p - e0]; }, [](int, int, uint64_t, int) {});
        wave_sync();
        if (k < 0) bad = true;
        else most = k > most ? k : most;
    }
    if ((threadIdx.x & 63) == 0) {   // one atomic per wave would serialise: 16 k of them took 200 us
        if (most > __hip_atomic_load(&info[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(&info[0], most);
        if (bad) atomicOr(&info[1], 1);
    }
}

// A wave per block; lds: 64 K values, then 64 K columns.
template <typename T>
__global__ __launch_bounds__(64) void k_sdia_fill(long nsl, int rows, int K, const int* __restrict__ rp,
                                                  const int* __restrict__ col, const T* __restrict__ val,
                                                  int* __restrict__ off, uint64_t* __restrict__ mask, T* __restrict__ out)
{
    extern __shared__ double lds[];
    T* const lv = reinterpret_cast<T*>(lds);
    int* const lc = reinterpret_cast<int*>(lv + 64 * K);
    const int lane = threadIdx.x;
    for (long sl = blockIdx.x; sl < nsl; sl += gridDim.x) {
        const long r0 = sl * 64, r1 = r0 + 64 < rows ? r0 + 64 : rows;
        const int e0 = rp[r0], ne = rp[r1] - e0;   // at most 64 K (k_sdia_count)
        wave_stage(col + e0, ne, lc);
        wave_stage(val + e0, ne, lv);
        wave_sync();
        auto put = [&](int k, int d, uint64_t m, int p) {
            out[(sl * K + k) * 64 + lane] = p >= 0 ? lv[p - e0] : T(0);
            if (lane == 0) {
                off[sl * K + k] = d;
                mask[sl * K + k] = m;
            }
        };
        const int n = walk_slice(r0, r1, rp, [&](int p) { return lc[p - e0]; }, put);
        for (int k = n < 0 ? 0 : n; k < K; ++k) put(k, 0, 0, -1);
        wave_sync();   // the next slice overwrites the areas
    }
}

// One row per lane: the row's product with x accumulated into (s, c), which may start
// from a first term (b of a residual, with NEG).  sl and K are wave-uniform; lanes past
// the last row hold no entry in any mask and pass any valid row as r.  KT > 0: A.K, known
// to the compiler; else eight diagonals at a time.  NC: sums of a row.
template <typename T, bool COMP, bool NEG, bool NT, int KT = 0, int NC = 2>
__device__ __forceinline__ void row(const sdia_view<T>& A, long sl, long r, const T* __restrict__ x, T& s, T& c)
{
    const int lane = threadIdx.x & 63;
    constexpr int CH = KT > 0 ? KT : 8;
    const int K = KT > 0 ? KT : A.K;
    const int* __restrict__ off = A.off + sl * K;
    const uint64_t* __restrict__ mask = A.mask + sl * K;
    const T* __restrict__ val = A.val + sl * K * 64 + lane;
    if constexpr (NC > 2) {
        static_assert(!COMP && KT == 0 && (NC == 4 || NC == 8 || NC == 16), "sd::row: plain rows");
        T acc[NC];
#pragma unroll
        for (int k = 0; k < NC; ++k) acc[k] = k == 0 ? s : T(0);
        for (int k0 = 0; k0 < K; k0 += CH) {
            T v[CH], xv[CH];
            bool on[CH];
            const int nk = K - k0;
#pragma unroll
            for (int k = 0; k < CH; ++k)
                if (k < nk) {
                    v[k] = NT ? dev::load_nt<T>(val + (long)(k0 + k) * 64) : val[(long)(k0 + k) * 64];
                    on[k] = ((mask[k0 + k] >> lane) & 1) != 0;
                    xv[k] = x[on[k] ? r + off[k0 + k] : r];
                }
#pragma unroll
            for (int k = 0; k < CH; ++k)
                if (k < nk) {
                    const T t = dev::fma_rn<T>(NEG ? -v[k] : v[k], xv[k], acc[k % NC]);
                    acc[k % NC] = on[k] ? t : acc[k % NC];
                }
            if (NC == 16) {   // the next eight diagonals go to the other eight sums
#pragma unroll
                for (int k = 0; k < CH; ++k) {
                    const T t = acc[k];
                    acc[k] = acc[(k + CH) % NC];
                    acc[(k + CH) % NC] = t;
                }
            }
        }
#pragma unroll
        for (int m = NC / 2; m >= 1; m >>= 1)
#pragma unroll
            for (int k = 0; k < NC / 2; ++k)
                if (k < m) acc[k] = acc[k] + acc[k + m];
        s = acc[0];
        return;
    }
    // (s, c): the sum the next entry goes to, (so, co): the other one
    T so = T(0), co = T(0);
    bool odd = false;
    for (int k0 = 0; k0 < K; k0 += CH) {
        T v[CH], xv[CH];
        bool on[CH];
        const int nk = K - k0;
#pragma unroll
        for (int k = 0; k < CH; ++k)
            if (KT > 0 || k < nk) {
                v[k] = NT ? dev::load_nt<T>(val + (long)(k0 + k) * 64) : val[(long)(k0 + k) * 64];
                on[k] = ((mask[k0 + k] >> lane) & 1) != 0;
                xv[k] = x[on[k] ? r + off[k0 + k] : r];
            }
#pragma unroll
        for (int k = 0; k < CH; ++k)
            if (KT > 0 || k < nk) {
                const T a = NEG ? -v[k] : v[k];
                T ns = s, nc = c;
                if (COMP) dev::dot2_step<T>(ns, nc, a, xv[k]);
                else ns = dev::fma_rn<T>(a, xv[k], ns);
                if (on[k]) {
                    s = so;
                    so = ns;
                    if (COMP) {
                        c = co;
                        co = nc;
                    }
                    odd = !odd;
                }
            }
    }
    if (COMP) {
        // entries 0, 2, ... first, as lane 0 of two merges lane 1's sum into its own
        T s1 = so, c1 = co;
        if (odd) {
            s1 = s;
            c1 = c;
            s = so;
            c = co;
        }
        dev::merge<T>(s, c, s1, c1);
    } else {
        s = s + so;
    }
}

}  // namespace sd
}  // namespace hpb
