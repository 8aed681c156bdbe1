// Tomogram: view_rt = sum_{d: P > 1e-6} P_dr K_dt / psum_r (update_tomogram_nobg,
// dragonfly/src/max_update.c:142-230), gathered per pixel over its frames.
//
// Two kernels per orientation chunk:
//  * posterior_rows_kernel copies the chunk's posterior into tiles whose rows are one 128-byte
//    line (16 FP64 or 32 FP32 orientations), rows[tile][frame][16 | 32], with every value the
//    tomogram leaves out (P <= 1e-6, or not a number) set to zero, and marks the rows that hold
//    anything, a bit a frame (counted by count_marks_kernel);
//  * tomogram_rows_kernel: block = one unit of pixels (at most 64 consecutive engine pixels and
//    about kTomoUnitEntries photons, tomo_units) x one such tile. The unit's photon list (pixels
//    ascending, frames ascending) is cut into 32 equal pieces, one for each stream of 8 lanes (8
//    streams a wavefront); a stream adds count * P row after row and adds its running sums into
//    the block's LDS tile when its piece passes to the next pixel. The tile is then divided by
//    psum and written orientation-major, or tile-major for the voxel-box merge and the pair
//    tomogram. A tile whose marked rows are at most half of the frames (late iterations: a
//    frame's posterior sits in a few orientations) is done by its marked rows alone: a wavefront
//    tests 64 entries of its quarter of the list at once and queues those whose row is marked.
// Why: a pixel's frames are spread over the whole data set, so rows are only read at L2 speed
// while the XCD's 4 MB L2 holds the tile's rows of every frame: 128 bytes a frame, where the
// 64-orientation rows of the posterior itself need 512 (and 128-byte pieces of those would use a
// quarter of the L2's sets). More than kFramesPerTomoRange frames take several launches, each adding to
// the view of the one before (as many as option tomo_parts allows, then with more frames each). Equal pieces of a unit's list
// and units of bounded photons, because pixels differ a thousandfold in photons (the 64 brightest
// can hold a quarter of all): a block that takes several times a tile's time lets the XCD go on to
// further tiles, whose rows then share its L2. Before, eight frame ranges wrote eight partial
// views of 64-orientation tiles that a second kernel added up: 30,000 frames x 10,880
// orientations of 186 photons (66,820 pixels) took 49.5 + 13.7 ms, now 29.7;
// 20,000 x 6300 on the 151 x 151 detector 8.9 + 2.8 ms, now 6.7 (11.1 without the bound on a
// unit's photons, 6.5 and 6.7 at 4096 and 8192); 4 rows in flight instead of 8 cost 2-4%.
#include <algorithm>
#include <vector>

#include "emc_common.h"
#include "emc_gather.h"
#include "emc_kernels.h"

namespace emc {

// One wave copies one frame's 64-orientation row at a time; block = 64 frames x 64 orientations.
template <typename T>
__global__ __launch_bounds__(kBlock) void posterior_rows_kernel(const double *__restrict__ P, int num_data, int r0,
                                                                int num_rot, T *__restrict__ rows,
                                                                unsigned long long *__restrict__ marks) {
    constexpr int W = kTomoRowBytes / sizeof(T), kTiles = kRTile / W;
    __shared__ unsigned long long s_mark[kTiles];
    if (threadIdx.x < kTiles) s_mark[threadIdx.x] = 0ull;
    __syncthreads();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int c = blockIdx.y * kRTile + lane;
    const bool real = r0 + c < num_rot;
    const double *__restrict__ src = P + (size_t)((r0 >> 6) + blockIdx.y) * num_data * kRTile + lane;
    T *__restrict__ dst = rows + (size_t)(c / W) * num_data * W + c % W;
    const int d1 = min(num_data, (int)(blockIdx.x + 1) * 64);
    unsigned long long mark = 0ull;  // of tile lane % kTiles
    for (int d = blockIdx.x * 64 + wave; d < d1; d += kWavesPerBlock) {
        const T p = (T)src[(size_t)d * kRTile];
        const bool keep = real && (double)p > kProbMin;
        dst[(size_t)d * W] = keep ? p : (T)0;
        const unsigned long long any = __ballot(keep) >> (lane % kTiles * W) & ((1ull << W) - 1ull);
        mark |= (unsigned long long)(any != 0ull) << (d % 64);
    }
    if (lane < kTiles) atomicOr(&s_mark[lane], mark);
    __syncthreads();
    if (threadIdx.x < kTiles)
        marks[((size_t)blockIdx.y * kTiles + threadIdx.x) * (gridDim.x + 1) + blockIdx.x] = s_mark[threadIdx.x];
}

// The number of marked rows of every tile, behind its marks; a wave a tile.
__global__ __launch_bounds__(kBlock) void count_marks_kernel(unsigned long long *__restrict__ marks, int words,
                                                             int ntiles) {
    const int tile = blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (tile >= ntiles) return;
    unsigned long long *__restrict__ m = marks + (size_t)tile * (words + 1);
    int count = 0;
    for (int i = lane; i < words; i += 64) count += __popcll(m[i]);
    for (int o = 32; o > 0; o >>= 1) count += __shfl_xor(count, o);
    if (lane == 0) m[words] = count;
}

template <typename T, typename OT, bool kRmajor>
__global__ __launch_bounds__(kBlock) void tomogram_rows_kernel(
    const T *__restrict__ rows, int num_data, int ntiles, const int2 *__restrict__ units, int num_units,
    const long *__restrict__ toff, const int *__restrict__ tframe, const double *__restrict__ tcnt, int num_pix,
    const unsigned long long *__restrict__ marks, int accumulate,
    const double *__restrict__ psum, int num_psum, OT *__restrict__ view) {
    using V = typename RowVec<T>::type;
    constexpr int n = RowVec<T>::n, W = kTomoRowBytes / sizeof(T);
    constexpr int LR = W / n, kStreams = kBlock / LR;  // a batch: LR entries, one staged by each lane of a stream
    __shared__ double s_sum[W][65];
    __shared__ RowEntry s_list[kWavesPerBlock][64];
    __shared__ int2 s_queue[kWavesPerBlock][128];  // marked entries: frame, place in the list
    __shared__ int s_off[65];
    // XCD-aware order: XCD x takes tiles x, x + kNumXcd, ... one at a time, every unit of a tile
    // together, so its L2 holds the rows of one tile
    const int tile = blockIdx.x % kNumXcd + kNumXcd * (int)(blockIdx.x / kNumXcd / num_units);
    if (tile >= ntiles) return;
    const int2 unit = units[blockIdx.x / kNumXcd % num_units];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int t0 = unit.x, nt = unit.y;  // 1 <= nt <= 64 pixels
    const long e0 = toff[t0];
    if (tid <= nt) s_off[tid] = (int)(toff[t0 + tid] - e0);
    for (int i = tid; i < W * 65; i += kBlock) (&s_sum[0][0])[i] = 0.;
    __syncthreads();
    const int total = s_off[nt];
    const int c = lane % LR, g = lane / LR;
    const T *__restrict__ col = rows + (size_t)tile * num_data * W + c * n;
    const int *__restrict__ frames = tframe + e0;
    const double *__restrict__ counts = tcnt + e0;
    const int words = (num_data + 63) / 64;
    const unsigned long long *__restrict__ mark = marks + (size_t)tile * (words + 1);
    const int marked = (int)mark[words];
    // by marks up to half of the frames: with 5.8% of the rows marked the tomogram of 15,013 frames x
    // 10,880 orientations (late posteriors) takes 5.4 ms, 17.4 by whole lists; with 27% 0.48 and 0.70 (2111
    // x 6480); with all 51 and 29.7 (30,000 x 10,880): the lines cross at about 52%
    if (2L * marked <= num_data) {
        const int quarter = (total + kWavesPerBlock - 1) / kWavesPerBlock;
        const int k1 = marked ? min(total, (wave + 1) * quarter) : 0;
        int2 *__restrict__ queue = s_queue[wave];
        int held = 0;
        // the first m <= 64 queued entries: a lane finds the pixel and count of one, then the
        // streams add 64 / LR rows at a time
        auto drain = [&](int m) {
            __builtin_amdgcn_wave_barrier();
            int2 e = make_int2(0, 0);
            if (lane < m) {
                e = queue[lane];
                int t = 0;
                for (int step = 32; step > 0; step >>= 1)
                    if (t + step < nt && s_off[t + step] <= e.y) t += step;
                e.y = (int)counts[e.y] * 64 | t;
            }
            V v[LR];
            int code[LR];
#pragma unroll
            for (int u = 0; u < LR; ++u) {
                const int i = u * (64 / LR) + g;
                const int frame = __shfl(e.x, i);
                code[u] = __shfl(e.y, i);
                v[u] = *reinterpret_cast<const V *>(col + (size_t)(unsigned)frame * W);
            }
#pragma unroll
            for (int u = 0; u < LR; ++u)
#pragma unroll
                for (int i = 0; i < n; ++i)
                    if (code[u] >= 64 && (double)v[u][i] != 0.)
                        unsafeAtomicAdd(&s_sum[c * n + i][code[u] % 64], (double)(code[u] / 64) * (double)v[u][i]);
            __builtin_amdgcn_wave_barrier();
        };
        constexpr int kTests = 4;
        for (int kb = wave * quarter; kb < k1; kb += kTests * 64) {
            int f[kTests];
            bool on[kTests];
#pragma unroll
            for (int u = 0; u < kTests; ++u) {
                const int k = kb + u * 64 + lane;
                f[u] = k < k1 ? frames[k] : -1;
            }
#pragma unroll
            for (int u = 0; u < kTests; ++u) on[u] = f[u] >= 0 && mark[f[u] / 64] >> (f[u] % 64) & 1ull;
#pragma unroll
            for (int u = 0; u < kTests; ++u) {
                const unsigned long long in = __ballot(on[u]);
                if (on[u]) queue[held + __popcll(in & ((1ull << lane) - 1ull))] = make_int2(f[u], kb + u * 64 + lane);
                held += __popcll(in);
                if (held >= 64) {
                    drain(64);
                    held -= 64;
                    if (lane < held) queue[lane] = queue[64 + lane];
                }
            }
        }
        if (held) drain(held);
    } else {
        const int per = (total + kStreams - 1) / kStreams;
        int k = min(total, (wave * (64 / LR) + g) * per);
        const int k_end = min(total, k + per);
        // the stream's first pixel: the last one whose list starts at or before k
        int t = 0;
        for (int step = 32; step > 0; step >>= 1)
            if (t + step < nt && s_off[t + step] <= k) t += step;
        int t_end = s_off[t + 1];
        double acc[n] = {};
        auto flush = [&] {
#pragma unroll
            for (int i = 0; i < n; ++i) {
                unsafeAtomicAdd(&s_sum[c * n + i][t], acc[i]);
                acc[i] = 0.;
            }
        };
        const int batches = (per + LR - 1) / LR;  // the same for every stream
        for (int b = 0; b < batches; ++b, k += LR) {
            // entries past the piece's end count nothing and read the (finite) row of frame 0
            RowEntry q{0, 0.f};
            if (k + c < k_end) q = RowEntry{frames[k + c], (float)counts[k + c]};
            s_list[wave][lane] = q;
            __builtin_amdgcn_wave_barrier();
            V v[LR];
            double w[LR];
#pragma unroll
            for (int u = 0; u < LR; ++u) {
                const RowEntry e = s_list[wave][g * LR + u];
                w[u] = (double)e.count;
                v[u] = *reinterpret_cast<const V *>(col + (size_t)(unsigned)e.row * W);
            }
            if (__all(min(k + LR, k_end) <= t_end)) {
#pragma unroll
                for (int u = 0; u < LR; ++u)
#pragma unroll
                    for (int i = 0; i < n; ++i) acc[i] += w[u] * (double)v[u][i];
            } else {
#pragma unroll
                for (int u = 0; u < LR; ++u) {
                    if (k + u < k_end && k + u >= t_end) {
                        flush();
                        while (k + u >= t_end) t_end = s_off[++t + 1];
                    }
#pragma unroll
                    for (int i = 0; i < n; ++i) acc[i] += w[u] * (double)v[u][i];
                }
            }
            __builtin_amdgcn_wave_barrier();  // the entries are read before the next batch replaces them
        }
        flush();
    }
    __syncthreads();
    // psum (nullable: sums only) of the tile's columns; columns past num_psum are padding
    const int c0 = tile * W;
    auto value = [&](int j, int i, size_t at) {
        double a = s_sum[j][i];
        if (accumulate) a += (double)view[at];
        const double ps = psum && c0 + j < num_psum ? psum[c0 + j] : 0.;
        return (OT)(ps > 0. ? a / ps : a);
    };
    if constexpr (kRmajor) {
        if (lane < nt)
            for (int j = wave; j < W; j += kWavesPerBlock) {
                const size_t at = (size_t)(c0 + j) * num_pix + t0 + lane;
                view[at] = value(j, lane, at);
            }
    } else {
        OT *__restrict__ base = view + (size_t)(c0 / kRTile) * num_pix * kRTile + c0 % kRTile;
        for (int i = tid; i < nt * W; i += kBlock) {
            const int p = i / W, j = i % W;
            const size_t at = (size_t)(base - view) + (size_t)(t0 + p) * kRTile + j;
            view[at] = value(j, p, at);
        }
    }
}

template <typename T>
static void rows_launch(hipStream_t s, const double *P, int num_data, int r0, int C, int num_rot, T *rows,
                        unsigned long long *marks) {
    if (num_data <= 0 || C <= 0) return;
    posterior_rows_kernel<T><<<dim3((num_data + 63) / 64, C / kRTile), kBlock, 0, s>>>(P, num_data, r0, num_rot, rows,
                                                                                        marks);
    const int ntiles = C / (int)(kTomoRowBytes / sizeof(T));
    count_marks_kernel<<<(ntiles + kWavesPerBlock - 1) / kWavesPerBlock, kBlock, 0, s>>>(marks, (num_data + 63) / 64, ntiles);
}

void launch_posterior_rows(hipStream_t s, const double *P, int num_data, int r0, int C, int num_rot, double *rows,
                           unsigned long long *marks) {
    rows_launch(s, P, num_data, r0, C, num_rot, rows, marks);
}

void launch_posterior_rows(hipStream_t s, const double *P, int num_data, int r0, int C, int num_rot, float *rows,
                           unsigned long long *marks) {
    rows_launch(s, P, num_data, r0, C, num_rot, rows, marks);
}

// Every frame range in turn (range x's list of pixel t: toff[x * num_pix + t] up to the next
// offset); the last one divides by psum.
template <typename T, typename OT>
static void tomogram_launch(hipStream_t s, const T *rows, const unsigned long long *marks, int num_data, int C,
                            const TomoLists &l, int num_pix,
                            const double *psum, int num_psum, OT *view, bool rmajor) {
    constexpr int W = kTomoRowBytes / sizeof(T);
    // columns of one launch: its blocks x kBlock work-items must fit the 32-bit grid size
    const long most = std::max(1L, ((1L << 24) - 1) / ((long)kNumXcd * l.num_units)) * kNumXcd * W;
    for (long c = 0; c < C; c += most) {
        const int cols = (int)std::min<long>(most, C - c), ntiles = cols / W;
        const unsigned grid = (unsigned)((long)kNumXcd * l.num_units * ((ntiles + kNumXcd - 1) / kNumXcd));
        const T *src = rows + (size_t)c * num_data;
        const unsigned long long *bits = marks + (size_t)(c / W) * ((num_data + 63) / 64 + 1);
        OT *dst = view + (size_t)c * num_pix;
        for (int x = 0; x < l.nparts; ++x) {
            const double *ps = psum && x == l.nparts - 1 ? psum + c : nullptr;
            const long *toff = l.off + (size_t)x * num_pix;
            const int valid = (int)std::max<long>(0, num_psum - c);
            if (rmajor)
                tomogram_rows_kernel<T, OT, true><<<grid, kBlock, 0, s>>>(
                    src, num_data, ntiles, l.units, l.num_units, toff, l.frame, l.cnt, num_pix, bits, x > 0, ps,
                    valid, dst);
            else
                tomogram_rows_kernel<T, OT, false><<<grid, kBlock, 0, s>>>(
                    src, num_data, ntiles, l.units, l.num_units, toff, l.frame, l.cnt, num_pix, bits, x > 0, ps,
                    valid, dst);
        }
    }
}

void launch_tomogram_rows(hipStream_t s, const double *rows, const unsigned long long *marks, int num_data, int C,
                          const TomoLists &l, int num_pix,
                          const double *psum, int num_psum, double *view, bool rmajor) {
    tomogram_launch(s, rows, marks, num_data, C, l, num_pix, psum, num_psum, view, rmajor);
}

void launch_tomogram_rows(hipStream_t s, const float *rows, const unsigned long long *marks, int num_data, int C,
                          const TomoLists &l, int num_pix,
                          const double *psum, int num_psum, double *view, bool rmajor) {
    tomogram_launch(s, rows, marks, num_data, C, l, num_pix, psum, num_psum, view, rmajor);
}

void launch_tomogram_rows(hipStream_t s, const float *rows, const unsigned long long *marks, int num_data, int C,
                          const TomoLists &l, int num_pix,
                          float *sums) {
    tomogram_launch(s, rows, marks, num_data, C, l, num_pix, nullptr, 0, sums, false);
}

// Units of pixels over the lists of nparts frame ranges (off as TomoLists::off, on the host):
// whole 64-pixel patches, cut after a pixel where they pass kTomoUnitEntries photons a range.
std::vector<int2> tomo_units(const long *off, int nparts, int num_pix) {
    std::vector<int2> units;
    for (int p0 = 0; p0 < num_pix; p0 += 64) {
        const int p1 = std::min(num_pix, p0 + 64);
        long held = 0;
        int first = p0;
        for (int t = p0; t < p1; ++t) {
            for (int x = 0; x < nparts; ++x) held += off[(size_t)x * num_pix + t + 1] - off[(size_t)x * num_pix + t];
            if (held >= (long)kTomoUnitEntries * nparts || t + 1 == p1) {
                units.push_back(make_int2(first, t + 1 - first));
                first = t + 1;
                held = 0;
            }
        }
    }
    return units;
}

}  // namespace emc
