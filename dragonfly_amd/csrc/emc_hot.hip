// Likelihood with the brightest pixels' rows in LDS: G_dr = sum_t K_dt log W_rt over one frame's
// photons (mask < 1), as likelihood_rows_kernel, for all frames of a data set.
//
// The gather is bound by what an XCD's L2 delivers (23.6 TB/s of rows chip-wide, 38 bytes a cycle and
// CU), while a CU's LDS delivers 128 bytes a cycle beside it; and photons crowd into few pixels: of 30,000
// frames of 187 photons on 66,820 pixels the brightest 256 hold 19%, of 100-photon frames on 22,801 pixels
// 53%. A block (16 waves, one a CU) therefore keeps the rows of up to kHotRows brightest pixels of one
// log W tile in LDS and serves a part of the frames: a wave takes a frame, gathers its other photons'
// rows through L2 and the bright ones' from LDS. The photon lists are split once per data set.
// Against the rows through L2 alone, ms: 30,000 frames of 187 photons x 10,880 orientations (66,820 pixels)
// 21.4 -> 19.6, 15,013 of 249 (38,190) 13.4 -> 11.3, 20,000 of 99 x 6300 (22,801) 4.0 -> 2.8, 2111 of 110 x 6480
// (7905) 0.50 -> 0.38, 3000 of 85 x 3240 0.34 -> 0.29; FP32 rows, 40,000 of 187 x 10,880: 15.7 -> 14.9. Rows of 128
// bytes, four times as many, were slower (24.5 and 6.5 for the first and third): their additions over
// eight streams and their lists cost more vector instructions than the loads. 136 rows: 19.6, 11.6, 2.75.
#include "emc_common.h"
#include "emc_gather.h"
#include "emc_kernels.h"

namespace emc {

constexpr int kHotThreads = 1024, kHotWaves = kHotThreads / 64;
constexpr int kHotRowBytes = 512;

// Each frame's likelihood list as entries: the photons of other pixels first, {pixel, count}, up to
// mid[d], then those of bright ones, {slot, count}. One wave a frame.
__global__ __launch_bounds__(kBlock) void hot_lists_kernel(const long *__restrict__ off, const int *__restrict__ pix,
                                                           const double *__restrict__ cnt,
                                                           const int *__restrict__ slot, int num_data,
                                                           RowEntry *__restrict__ entry, long *__restrict__ mid) {
    const int lane = threadIdx.x & 63, d = blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
    if (d >= num_data) return;
    const long k1 = off[d + 1];
    long front = off[d], back = k1;
    for (long kb = off[d]; kb < k1; kb += 64) {
        const long k = kb + lane;
        const bool in = k < k1;
        const int p = in ? pix[k] : 0, h = in ? slot[p] : -1;
        const unsigned long long cold = __ballot(in && h < 0), hot = __ballot(h >= 0);
        const unsigned long long below = (1ull << lane) - 1ull;
        if (in) {
            const float c = (float)cnt[k];
            if (h < 0) entry[front + __popcll(cold & below)] = RowEntry{p, c};
            else entry[back - 1 - __popcll(hot & below)] = RowEntry{h, c};
        }
        front += __popcll(cold);
        back -= __popcll(hot);
    }
    if (lane == 0) mid[d] = front;
}

// acc += count x row over m <= 64 staged entries, S of them at once, up to U steps in flight; row(r)
// gives the lane's 16 bytes of row r
template <typename T, int S, int U, typename Row>
__device__ __forceinline__ void add_steps(const RowEntry *list, int &s, int m, int g, double (&acc)[RowVec<T>::n],
                                          Row &&row) {
    constexpr int n = RowVec<T>::n;
    for (; s + S * U <= m; s += S * U) {
        typename RowVec<T>::type v[U];
        float w[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const RowEntry q = list[s + u * S + g];
            w[u] = q.count;
            v[u] = row(q.row);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < n; ++i) acc[i] += (double)w[u] * (double)v[u][i];
    }
}

template <typename T, int S, typename Row>
__device__ __forceinline__ void add_staged(const RowEntry *list, int m, int g, double (&acc)[RowVec<T>::n], Row &&row) {
    int s = 0;
    add_steps<T, S, 8>(list, s, m, g, acc, row);
    add_steps<T, S, 4>(list, s, m, g, acc, row);
    add_steps<T, S, 2>(list, s, m, g, acc, row);
    add_steps<T, S, 1>(list, s, m, g, acc, row);
    if (s + g < m) {
        const RowEntry q = list[s + g];
        const typename RowVec<T>::type v = row(q.row);
#pragma unroll
        for (int i = 0; i < RowVec<T>::n; ++i) acc[i] += (double)q.count * (double)v[i];
    }
}

// kW: orientations of a log W tile (64 FP64, 128 FP32)
template <typename T, int kW>
__global__ __launch_bounds__(kHotThreads) void likelihood_hot_kernel(
    const T *__restrict__ logw, int C, int ntiles, int num_pix, const int *__restrict__ hot, int num_hot,
    const long *__restrict__ off, const long *__restrict__ mid, const RowEntry *__restrict__ entry,
    const uint8_t *__restrict__ blacklist, int num_data, int nparts, double *__restrict__ G, size_t tsG, int r0) {
    using V = typename RowVec<T>::type;
    constexpr int n = RowVec<T>::n, LR = kW / n, S = 64 / LR;
    extern __shared__ __align__(16) char hot_smem[];
    T *s_hot = reinterpret_cast<T *>(hot_smem);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    RowEntry *list = reinterpret_cast<RowEntry *>(hot_smem + (size_t)num_hot * kHotRowBytes) + wave * 64;
    // XCD x takes tiles x, x + kNumXcd, ... one at a time, every part of the frames together
    const int j = blockIdx.x / kNumXcd, part = j % nparts, tile = blockIdx.x % kNumXcd + kNumXcd * (j / nparts);
    if (tile >= ntiles) return;
    const int c = lane % LR * n, g = lane / LR;
    const T *__restrict__ col = logw + (size_t)tile * num_pix * kW + c;
    for (int i = tid / LR; i < num_hot; i += kHotThreads / LR)
        *reinterpret_cast<V *>(s_hot + i * kW + c) = *reinterpret_cast<const V *>(col + (size_t)hot[i] * kW);
    __syncthreads();
    const int r = tile * kW + c;
    auto cold_row = [&](int p) { return *reinterpret_cast<const V *>(col + (size_t)(unsigned)p * kW); };
    auto hot_row = [&](int h) { return *reinterpret_cast<const V *>(s_hot + h * kW + c); };
    // a wave takes consecutive frames of the part, 64 of them at a time: their bounds a lane each, the
    // first 64 entries of either kind of the next frame on their way while one is gathered
    const long d0 = (long)num_data * part / nparts, nd = (long)num_data * (part + 1) / nparts - d0;
    const long dw1 = d0 + nd * (wave + 1) / kHotWaves;
    for (long db = d0 + nd * wave / kHotWaves; db < dw1; db += 64) {
        const long d = min(db + lane, (long)num_data - 1), base = off[db];
        const int b0 = (int)(off[d] - base), bm = (int)(mid[d] - base), b1 = (int)(off[d + 1] - base);
        unsigned long long todo = __ballot(db + lane < dw1 && !blacklist[d]);
        const RowEntry *__restrict__ ent = entry + base;
        auto fetch = [&](int k, int k1) { return k + lane < k1 ? ent[k + lane] : RowEntry{0, 0.f}; };
        if (!todo) continue;
        int f = __ffsll((long long)todo) - 1;
        int k0 = __builtin_amdgcn_readlane(b0, f), km = __builtin_amdgcn_readlane(bm, f), k1 = __builtin_amdgcn_readlane(b1, f);
        RowEntry cold = fetch(k0, km), hot_e = fetch(km, k1);
        while (todo) {
            todo &= todo - 1ull;
            const int f2 = todo ? __ffsll((long long)todo) - 1 : f;
            const int n0 = __builtin_amdgcn_readlane(b0, f2), nm = __builtin_amdgcn_readlane(bm, f2),
                      n1 = __builtin_amdgcn_readlane(b1, f2);
            double acc[n] = {};
            int k = k0;
            do {
                list[lane] = cold;
                const int m = min(64, km - k);
                k += 64;
                cold = k < km ? fetch(k, km) : fetch(n0, nm);
                __builtin_amdgcn_wave_barrier();
                add_staged<T, S>(list, m, g, acc, cold_row);
                __builtin_amdgcn_wave_barrier();  // the entries are read before the next replace them
            } while (k < km);
            k = km;
            do {
                list[lane] = hot_e;
                const int m = min(64, k1 - k);
                k += 64;
                hot_e = k < k1 ? fetch(k, k1) : fetch(nm, n1);
                __builtin_amdgcn_wave_barrier();
                add_staged<T, S>(list, m, g, acc, hot_row);
                __builtin_amdgcn_wave_barrier();
            } while (k < k1);
#pragma unroll
            for (int o = LR; o < 64; o <<= 1)
#pragma unroll
                for (int i = 0; i < n; ++i) acc[i] += __shfl_xor(acc[i], o);
            if (lane < LR && r < C)
                store_sums<n>(G + (size_t)((r0 + r) / kRTile) * tsG + (size_t)(db + f) * kRTile + r % kRTile, acc);
            f = f2, k0 = n0, km = nm, k1 = n1;
        }
    }
}

void launch_hot_lists(hipStream_t s, const long *off, const int *pix, const double *cnt, const int *slot, int num_data,
                      RowEntry *entry, long *mid) {
    if (num_data <= 0) return;
    hot_lists_kernel<<<(num_data + kWavesPerBlock - 1) / kWavesPerBlock, kBlock, 0, s>>>(off, pix, cnt, slot, num_data,
                                                                                        entry, mid);
}

template <typename T, int kW>
static void hot_launch(hipStream_t s, const T *logw, int C, int num_pix, const HotLists &h, const long *off,
                       const uint8_t *blacklist, int num_data, double *G, int r0) {
    if (num_data <= 0 || C <= 0) return;
    const int ntiles = (C + kW - 1) / kW;
    const size_t lds = (size_t)h.num * kHotRowBytes + kHotWaves * 64 * sizeof(RowEntry);
    const long per = (ntiles + kNumXcd - 1) / kNumXcd;
    int parts = h.parts;
    while (parts > 1 && kNumXcd * parts * per > 1L << 21) parts /= 2;  // work-items of a grid: 32 bits
    const unsigned grid = (unsigned)(kNumXcd * parts * per);
    likelihood_hot_kernel<T, kW><<<grid, kHotThreads, lds, s>>>(logw, C, ntiles, num_pix, h.pix, h.num, off, h.mid, h.entry,
                                                               blacklist, num_data, parts, G,
                                                               (size_t)num_data * kRTile, r0);
}

void launch_likelihood_hot(hipStream_t s, const double *logw, int C, int num_pix, const HotLists &h, const long *off,
                           const uint8_t *blacklist, int num_data, double *G, int r0) {
    hot_launch<double, kRTile>(s, logw, C, num_pix, h, off, blacklist, num_data, G, r0);
}

void launch_likelihood_hot(hipStream_t s, const float *logw, int C, int num_pix, const HotLists &h, const long *off,
                           const uint8_t *blacklist, int num_data, double *G, int r0) {
    hot_launch<float, 2 * kRTile>(s, logw, C, num_pix, h, off, blacklist, num_data, G, r0);
}

}  // namespace emc
