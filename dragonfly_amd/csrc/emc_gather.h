// Photon gathers: one wavefront's sum over a list of (row, count) entries of
// count * matrix[row][...], the inner loop of the likelihood (rows of log W, one per photon of
// a frame).
//
// A row is kRow consecutive elements (64 FP64 or 128 FP32 orientations, 512 bytes; a pair of a
// 128-wide FP32 row takes its 256-byte half). Each lane loads 16 bytes of a row, so LR lanes
// cover it and the wavefront walks S = 64 / LR entries of the list at once, U such steps in
// flight; the S partial sums are added at the end. The list is staged through LDS 64 entries at
// a time by one coalesced load, and read back as broadcasts. Bound: what the XCD's L2
// delivers. Against one 8-byte load per lane and entry with the list in scalar registers
// (30,000 frames x 10,880 orientations of 186 photons on 66,820 pixels, FP64): 26.8 -> 20.6 ms,
// 18.2 -> 23.6 TB/s of rows; U = 4 or 8 alike; 128-, 256- and 1024-byte rows 21.0, 19.2, 27.1 ms.
#pragma once

#include "emc_common.h"
#include "emc_kernels.h"

namespace emc {

// 16 bytes of a row
template <typename T>
struct RowVec;
template <>
struct RowVec<double> {
    static constexpr int n = 2;
    typedef double type __attribute__((ext_vector_type(2)));
};
template <>
struct RowVec<float> {
    static constexpr int n = 4;
    typedef float type __attribute__((ext_vector_type(4)));
};

// acc[i] += sum over entries k0 <= k < k1 of cnt[k] * col[idx[k] * kRow + i]; col is the lane's
// 16 bytes of row 0 (lane % LR), s_list the wavefront's 64 entries of LDS. On return every
// lane of a stream-aligned set holds the full sums of its columns.
template <typename T, int kRow, int LR, int U>
__device__ __forceinline__ void gather_rows(const T *__restrict__ col, const int *__restrict__ idx,
                                            const double *__restrict__ cnt, long k, long k1, RowEntry *s_list,
                                            int lane, double (&acc)[RowVec<T>::n]) {
    using V = typename RowVec<T>::type;
    constexpr int n = RowVec<T>::n, S = 64 / LR;
    const int g = lane / LR;
    for (; k < k1; k += 64) {
        const int m = (int)min((long)64, k1 - k);
        if (lane < m) s_list[lane] = RowEntry{idx[k + lane], (float)cnt[k + lane]};
        __builtin_amdgcn_wave_barrier();
        int s = 0;
        for (; s + S * U <= m; s += S * U) {
            V v[U];
            double c[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const RowEntry q = s_list[s + u * S + g];
                c[u] = (double)q.count;
                v[u] = *reinterpret_cast<const V *>(col + (size_t)(unsigned)q.row * kRow);
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int i = 0; i < n; ++i) acc[i] += c[u] * (double)v[u][i];
        }
        for (; s < m; s += S) {
            const int e = s + g;
            if (e < m) {
                const RowEntry q = s_list[e];
                const V v = *reinterpret_cast<const V *>(col + (size_t)(unsigned)q.row * kRow);
#pragma unroll
                for (int i = 0; i < n; ++i) acc[i] += (double)q.count * (double)v[i];
            }
        }
        __builtin_amdgcn_wave_barrier();  // the entries are read before the next 64 replace them
    }
#pragma unroll
    for (int o = LR; o < 64; o <<= 1)
#pragma unroll
        for (int i = 0; i < n; ++i) acc[i] += __shfl_xor(acc[i], o);
}

// Columns [c, c + n) of a 64-wide output row from the lanes of the first stream.
template <int n>
__device__ __forceinline__ void store_sums(double *dst, const double (&acc)[n]) {
#pragma unroll
    for (int i = 0; i < n; i += 2) *reinterpret_cast<double2 *>(dst + i) = make_double2(acc[i], acc[i + 1]);
}

}  // namespace emc
