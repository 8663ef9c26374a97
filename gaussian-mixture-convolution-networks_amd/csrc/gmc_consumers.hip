// Forward evaluations with the reductions of their callers fused in, for the two consumers that evaluate a mixture
// (given by its covariances) and reduce the values at once:
//   * ReLU transfer fitting by fixed-point iteration (src/gmc/fitting.py:287-312): the target mixture is evaluated
//     at the fitting mixture's own centres and turned into the goal relu(v + c) - relu(c); every iteration evaluates
//     the fitting mixture with the weights |x| at its centres and applies x <- |x| (goal + 0.05) / (v + 0.05);
//   * BatchNorm (src/gmc/modules.py:374-425): the mixture is evaluated at sampling positions and only the sum and the
//     count, mean and sum of squared deviations of (v + constant) per workgroup are kept (torch.std_mean of the
//     sampled values).
// The values never go to memory.  These shapes have few points per mixture (the 128 centres, 100 samples), so one
// workgroup covers all points of its mixture: the all-vector "4 x 16" layout of gmc_dense.hip with 64 P points per
// workgroup.  Also here: the optional input check of the reference's CUDA backward (util/mixture.h:85-93).
#include "gmc_common.h"

namespace gmc {

int check_shape(const gmc_shape* s);

constexpr int kTileC = 256;

enum { kEpiStore = 0, kEpiReluShift = 1, kEpiRatio = 2, kEpiMoments = 3 };

template <typename T> struct EpiArgs {
    const T* constant;     // [B][L]                     kinds 1, 3
    const T* goal;         // [B][L][N]                  kind 2
    const T* weights;      // [B][L][M], M == N          kind 2: x of the iteration, evaluated as |x|
    T* out;                // [B][L][N]                  kinds 0, 1, 2
    double* moments;       // [B L][chunks][3] count, mean, sum of squared deviations from that mean   kind 3
};

// points: point n of mixture bl is read from points[bl * mixture_stride + n * point_stride + d] (query tensor
// [B][L][N][D]: strides N D and D; the centres of a mixture [B][L][N][G]: pointer to its first position, strides N G
// and G).  `mixture` holds covariances.
template <typename T, int D, int P, int KIND>
__global__ __launch_bounds__(kBlock) void consumer_fwd_kernel(const T* __restrict__ mixture, const T* __restrict__ points,
                                                              size_t mixture_stride, int point_stride, EpiArgs<T> epi,
                                                              int L, int M, int N, int chunks, int n_mixtures) {
    constexpr int G = 1 + D + D * D;
    constexpr int S = Rec<T, D>::kStride;
    __shared__ __attribute__((aligned(16))) T lds[(kTileC + 6) * S];
    __shared__ int counts[10];
    __shared__ double wave_moments[4][2];
    const T* exp2_tab = exp2_table<T>();            // (published by the barriers of staging)

    int bl, chunk;
    map_workgroup(blockIdx.x, chunks, n_mixtures, bl, chunk);
    if (bl >= n_mixtures) return;
    const T* __restrict__ mix_bl = mixture + size_t(bl) * M * G;
    const T* __restrict__ x_bl = points + size_t(bl) * mixture_stride;

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row = lane >> 4, col = lane & 15;
    T x[P][D];
    T acc[P];
    const int n0 = (chunk * 4 + wave) * (16 * P) + col;
#pragma unroll
    for (int p = 0; p < P; ++p) {
        int n = n0 + p * 16;
        n = n < N ? n : N - 1;
#pragma unroll
        for (int d = 0; d < D; ++d) x[p][d] = x_bl[size_t(n) * point_stride + d];
        acc[p] = T(0);
    }
    for (int g0 = 0; g0 < M; g0 += kTileC) {
        const int cnt = (M - g0) < kTileC ? (M - g0) : kTileC;
        const T* over = KIND == kEpiRatio ? epi.weights + size_t(bl) * M + g0 : nullptr;
        stage_tile<T, D, 4>(mix_bl + size_t(g0) * G, cnt, 1.0, lds, counts, true, over);
        const int centred_start = counts[8], padded_total = counts[9];
        add_pairs<T, D, P, 4, false>(lds, exp2_tab, row, centred_start, x, acc);
        add_pairs<T, D, P, 4, true>(lds, exp2_tab, centred_start + row, padded_total, x, acc);
    }
    double vals[P];                                  // kind 3: this lane's values (rows other than 0 and points beyond N: none)
    double s1 = 0.0;
    int mine = 0;
#pragma unroll
    for (int p = 0; p < P; ++p) {
        vals[p] = 0.0;
        T v = acc[p];
        v += __shfl_xor(v, 16, 64);
        v += __shfl_xor(v, 32, 64);
        const int n = n0 + p * 16;
        if (row == 0 && n < N) {
            const size_t at = size_t(bl) * N + n;
            if constexpr (KIND == kEpiReluShift) {
                const T c = epi.constant[bl];
                const T shifted = v + c;
                epi.out[at] = (shifted > T(0) ? shifted : T(0)) - (c > T(0) ? c : T(0));
            } else if constexpr (KIND == kEpiRatio) {
                const T xw = epi.weights[at];                       // M == N: point n is the centre of component n
                epi.out[at] = (xw < T(0) ? -xw : xw) * (epi.goal[at] + T(0.05)) / (v + T(0.05));
            } else {
                vals[p] = double(v) + double(epi.constant[bl]);
                s1 += vals[p];
                mine |= 1 << p;
            }
        }
    }
    if constexpr (KIND == kEpiMoments) {
        // Two passes over the values the workgroup holds in registers: their mean, then the squared deviations from
        // it.  (Sum and sum of squares in one pass lose (mean / sd)^2 ulps of the variance: a large constant with a
        // small spread of the values, as BatchNorm meets it behind a large bias, came out as noise.)
        const int here = (N - chunk * 64 * P) < 64 * P ? (N - chunk * 64 * P) : 64 * P;     // points of this workgroup
        s1 = wave_sum_to_lane63(s1);
        if (lane == 63) wave_moments[wave][0] = s1;
        __syncthreads();
        const double mean = ((wave_moments[0][0] + wave_moments[1][0]) + (wave_moments[2][0] + wave_moments[3][0])) / double(here);
        double m2 = 0.0;
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const double dv = vals[p] - mean;
            m2 += ((mine >> p) & 1) ? dv * dv : 0.0;
        }
        m2 = wave_sum_to_lane63(m2);
        if (lane == 63) wave_moments[wave][1] = m2;
        __syncthreads();
        if (threadIdx.x == 0) {
            double* o = epi.moments + (size_t(bl) * chunks + chunk) * 3;
            o[0] = double(here);
            o[1] = mean;
            o[2] = (wave_moments[0][1] + wave_moments[1][1]) + (wave_moments[2][1] + wave_moments[3][1]);
        }
    }
}

// The same for few points and many Gaussians (a layer's convolved mixtures at the 128 centres of the fitted ones or at
// 100 sampling positions).  The kernel above gives every wavefront a quarter of the points and all Gaussians: at 128
// points an LDS record serves two pairs of a lane, and all four wavefronts wait for the preparation of every tile.
// Here every wavefront holds ALL points (16 P, at most 256) and takes every fourth group of 64 Gaussians through its own
// LDS tile, without a barrier until the four partial values of a point are added at the end.  Kind 0 is the plain
// evaluation (gmc_dense.hip calls it), the only one with its Gaussians dealt to several workgroups (`ts`); its points
// may be shared by mixtures (Bx, Lx).
template <typename T, int D, int P, int KIND>
__global__ __launch_bounds__(kBlock) void few_points_fwd_kernel(const T* __restrict__ mixture, const T* __restrict__ points,
                                                                size_t mixture_stride, int point_stride, EpiArgs<T> epi,
                                                                int L, int M, int N, int Bx, int Lx, int n_mixtures,
                                                                bool covariance_form, TileSlices ts) {
    constexpr int G = 1 + D + D * D;
    constexpr int S = Rec<T, D>::kStride;
    constexpr int kWaves = kBlock / kWave;
    static_assert(KIND != kEpiRatio, "its points are as many as its components");
    static_assert(16 * P <= kBlock, "one lane per point at the end");
    constexpr int kWaveScalars = (kWave + 6) * S > 16 * P ? (kWave + 6) * S : 16 * P;
    __shared__ __attribute__((aligned(16))) T lds[kWaves * kWaveScalars];
    __shared__ double wave_moments[kWaves][2];
    const T* exp2_tab = exp2_table<T>();
    if constexpr (sizeof(T) == 8) __syncthreads();

    int bl, slice;
    map_workgroup(blockIdx.x, ts.slices, n_mixtures, bl, slice);
    if (bl >= n_mixtures) return;
    const int g_begin = slice * ts.per_slice;
    const int g_end = (g_begin + ts.per_slice) < M ? (g_begin + ts.per_slice) : M;
    const int b = bl / L, l = bl - b * L;
    const int xb = b < Bx ? b : Bx - 1, xl = l < Lx ? l : Lx - 1;
    const T* __restrict__ mix_bl = mixture + size_t(bl) * M * G;
    const T* __restrict__ x_bl = points + (size_t(xb) * Lx + xl) * mixture_stride;

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row = lane >> 4, col = lane & 15;
    T* tile = lds + wave * kWaveScalars;
    T x[P][D];
    T acc[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        int n = col + p * 16;
        n = n < N ? n : N - 1;
#pragma unroll
        for (int d = 0; d < D; ++d) x[p][d] = x_bl[size_t(n) * point_stride + d];
        acc[p] = T(0);
    }
    for (int g0 = g_begin + wave * kWave; g0 < g_end; g0 += kBlock) {
        const bool active = g0 + lane < g_end;
        const int m = active ? g0 + lane : g0;
        const Derived<D> dv = derive<T, D>(mix_bl + size_t(m) * G, covariance_form);
        const WaveTile t = stage_wave_tile<T, D, 4>(dv, active, 1.0, tile, lane);
        add_pairs<T, D, P, 4, false>(tile, exp2_tab, row, t.centred_start, x, acc);
        add_pairs<T, D, P, 4, true>(tile, exp2_tab, t.centred_start + row, t.padded_total, x, acc);
    }
    wave_fence();
#pragma unroll
    for (int p = 0; p < P; ++p) {
        T v = acc[p];
        v += __shfl_xor(v, 16, 64);
        v += __shfl_xor(v, 32, 64);
        if (row == 0) tile[col + p * 16] = v;
    }
    __syncthreads();
    const int n = threadIdx.x;
    const bool mine = n < N;
    T v = T(0);
    if (mine) v = (lds[n] + lds[kWaveScalars + n]) + (lds[2 * kWaveScalars + n] + lds[3 * kWaveScalars + n]);
    const size_t at = size_t(bl) * N + n;
    if constexpr (KIND == kEpiStore) {
        if (mine) { if (ts.slices > 1) atomic_add(&epi.out[at], v); else epi.out[at] = v; }
    } else if constexpr (KIND == kEpiReluShift) {
        if (mine) {
            const T c = epi.constant[bl];
            const T shifted = v + c;
            epi.out[at] = (shifted > T(0) ? shifted : T(0)) - (c > T(0) ? c : T(0));
        }
    } else {
        // mean, then squared deviations from it, of the workgroup's values (see the kernel above)
        const double value = mine ? double(v) + double(epi.constant[bl]) : 0.0;
        const double s1 = wave_sum_to_lane63(value);
        if (lane == 63) wave_moments[wave][0] = s1;
        __syncthreads();
        const double mean = ((wave_moments[0][0] + wave_moments[1][0]) + (wave_moments[2][0] + wave_moments[3][0])) / double(N);
        const double dv = value - mean;
        const double m2 = wave_sum_to_lane63(mine ? dv * dv : 0.0);
        if (lane == 63) wave_moments[wave][1] = m2;
        __syncthreads();
        if (threadIdx.x == 0) {
            double* o = epi.moments + size_t(bl) * 3;               // one record per mixture: one workgroup has all points
            o[0] = double(N);
            o[1] = mean;
            o[2] = (wave_moments[0][1] + wave_moments[1][1]) + (wave_moments[2][1] + wave_moments[3][1]);
        }
    }
}

// points per lane and workgroups per mixture for N points per mixture
static int consumer_points_per_lane(int N) { return N <= 128 ? 2 : N <= 256 ? 4 : 8; }
static int consumer_chunks(int N) { const int P = consumer_points_per_lane(N); return (N + 64 * P - 1) / (64 * P); }

// As few_points_fwd in gmc_dense.hip: more than two groups of Gaussians for the four wavefronts, three full ones above 96
// points, in double at most 96 points.  One workgroup has all points.  Kernel above / this one in us: 1600 mixtures of 5120
// Gaussians at 128 points 296 / 277; 50 x 129 at 122, 3-D, 6.6 / 7.3; float64 14 x 315 at 109 17.1 / 20.3, 3-D 3 x 166 at
// 103 11.6 / 13.6.
template <typename T> static bool few_points_consumer(int M, int N) {
    return M > 128 && (N <= 96 || (sizeof(T) == 4 && N <= 128 && M >= 192));
}

template <typename T, int D, int KIND>
static void launch_few_points(const T* mixture, const T* points, size_t mixture_stride, int point_stride, const EpiArgs<T>& epi,
                              int B, int L, int M, int N, int Bx, int Lx, bool cov, TileSlices ts, hipStream_t stream) {
    const size_t BL = size_t(B) * L;
    const dim3 grid(unsigned(grid_mixtures(BL) * ts.slices));
    const int P = (N + 15) / 16;
#define GMC_FEW(PP) few_points_fwd_kernel<T, D, PP, KIND><<<grid, dim3(kBlock), 0, stream>>>(mixture, points, mixture_stride, point_stride, epi, L, M, N, Bx, Lx, int(BL), cov, ts)
    // (the rules of the callers: at most 16 P = 64 points for the plain evaluation in double and 256 in float, 96 and 128
    // for the reductions)
    if (P <= 2) GMC_FEW(2); else if (P <= 4) GMC_FEW(4);
    else if constexpr (sizeof(T) == 4 || KIND != kEpiStore) {
        if (P <= 6) GMC_FEW(6);
        else if constexpr (sizeof(T) == 4) {
            if (P == 7) GMC_FEW(7); else if (P == 8) GMC_FEW(8);
            else if constexpr (KIND == kEpiStore) {
                if (P <= 10) GMC_FEW(10); else if (P <= 12) GMC_FEW(12); else if (P == 13) GMC_FEW(13); else GMC_FEW(16);
            }
        }
    }
#undef GMC_FEW
}

// The plain evaluation of mixtures with at most 256 points (gmc_dense.hip; `out` was cleared if there are slices).
void few_points_forward(const void* mixture, const void* xes, void* out, const gmc_shape& s, bool cov, TileSlices ts,
                        hipStream_t stream) {
#define GMC_GO(T, DD) do { EpiArgs<T> e{nullptr, nullptr, nullptr, (T*)out, nullptr}; \
        launch_few_points<T, DD, kEpiStore>((const T*)mixture, (const T*)xes, size_t(s.N) * DD, DD, e, s.B, s.L, s.M, s.N, s.Bx, s.Lx, cov, ts, stream); } while (0)
    if (s.dtype == GMC_F32) { if (s.D == 2) GMC_GO(float, 2); else GMC_GO(float, 3); }
    else { if (s.D == 2) GMC_GO(double, 2); else GMC_GO(double, 3); }
#undef GMC_GO
}

template <typename T, int D, int KIND>
static int launch_consumer(const T* mixture, const T* points, size_t mixture_stride, int point_stride, const EpiArgs<T>& epi,
                           int B, int L, int M, int N, hipStream_t stream) {
    const size_t BL = size_t(B) * L;
    if (BL == 0 || N == 0) return GMC_OK;
    if constexpr (KIND != kEpiRatio) {                  // (the ratio's points are the components themselves: not many against them)
        if (few_points_consumer<T>(M, N)) {
            launch_few_points<T, D, KIND>(mixture, points, mixture_stride, point_stride, epi, B, L, M, N, B, L, true,
                                          TileSlices{1, M}, stream);
            return hipGetLastError() == hipSuccess ? GMC_OK : GMC_E_LAUNCH;
        }
    }
    const int P = consumer_points_per_lane(N);
    const int chunks = consumer_chunks(N);
    if (grid_mixtures(BL) * chunks > max_workgroups(kBlock)) return GMC_E_SHAPE;
    const dim3 grid(unsigned(grid_mixtures(BL) * chunks));
#define GMC_CONS(PP) consumer_fwd_kernel<T, D, PP, KIND><<<grid, dim3(kBlock), 0, stream>>>(mixture, points, mixture_stride, point_stride, epi, L, M, N, chunks, int(BL))
    if (P == 2) GMC_CONS(2); else if (P == 4) GMC_CONS(4); else GMC_CONS(8);
#undef GMC_CONS
    return hipGetLastError() == hipSuccess ? GMC_OK : GMC_E_LAUNCH;
}

// (count, mean, sum of squared deviations) of the union of two sets of values (Chan, Golub, LeVeque 1979)
struct Moments { double n, mean, m2; };
__device__ __forceinline__ Moments merge_moments(const Moments& a, const Moments& b) {
    const double n = a.n + b.n;
    if (!(n > 0.0)) return Moments{0.0, 0.0, 0.0};
    const double delta = b.mean - a.mean, share = b.n / n;
    return Moments{n, a.mean + delta * share, a.m2 + b.m2 + delta * delta * a.n * share};
}

// sd (unbiased, as torch.std_mean) and mean of every slot from the workgroups' (count, mean, squared deviations):
// one wavefront per slot merges the records of the slot's workgroups (per_sample: the chunks of mixture `slot`;
// otherwise the chunks of layer `slot` in every batch entry), in a fixed order.  With running
// averages (BatchNorm in training, src/gmc/modules.py:405-410): they are updated in place by the factor alpha and take
// the place of the statistics.  inv_sd (optional) = 1 / max(sd, 0.001) (modules.py:414-415).
template <typename T>
__global__ __launch_bounds__(kBlock) void moments_finish_kernel(const double* __restrict__ moments, T* __restrict__ sd,
                                                                T* __restrict__ mean, T* __restrict__ inv_sd, T* running_sd,
                                                                T* running_mean, double alpha, int slots, int B, int L,
                                                                int chunks, int per_sample) {
    const int lane = threadIdx.x & 63;
    const int i = blockIdx.x * (kBlock / kWave) + (threadIdx.x >> 6);
    if (i >= slots) return;
    const int records = per_sample ? chunks : B * chunks;
    Moments acc{0.0, 0.0, 0.0};
    for (int r = lane; r < records; r += kWave) {
        const size_t bl = per_sample ? size_t(i) : size_t(r / chunks) * L + i;
        const double* rec = moments + (bl * chunks + (r % chunks)) * 3;
        acc = merge_moments(acc, Moments{rec[0], rec[1], rec[2]});
    }
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const Moments other{__shfl_xor(acc.n, off, kWave), __shfl_xor(acc.mean, off, kWave), __shfl_xor(acc.m2, off, kWave)};
        // both partners combine (lower lane, upper lane) in this order, so that they hold the same bits afterwards
        acc = (lane & off) ? merge_moments(other, acc) : merge_moments(acc, other);
    }
    if (lane != 0) return;
    const double var = acc.n > 1.0 ? acc.m2 / (acc.n - 1.0) : NAN;            // one value: undefined, as in torch
    T sd_i = T(sqrt(var));
    T mean_i = T(acc.mean);
    if (running_sd) {
        sd_i = T((1.0 - alpha) * double(running_sd[i]) + alpha * double(sd_i));
        mean_i = T((1.0 - alpha) * double(running_mean[i]) + alpha * double(mean_i));
        running_sd[i] = sd_i;
        running_mean[i] = mean_i;
    }
    sd[i] = sd_i;
    mean[i] = mean_i;
    if (inv_sd) inv_sd[i] = T(1) / (sd_i > T(0.001) ? sd_i : T(0.001));
}

// Sampling positions of BatchNorm (src/gmc/modules.py:394-400): the uniform numbers u [B][L][N][D] become positions in
// the box of all centres of batch entry b (over layers and components), widened in 2-D by u * 1.3 - 0.15.  The
// numbers of a batch entry are dealt to `chunks` workgroups, each of which finds the box itself (a second launch or a
// scratch buffer for the box would cost more).  Bound by the latency of reading the centres, which are many behind a
// convolution: sixteen wavefronts with eight centres per lane in flight (100 batch entries of 81920 centres: 177 us with
// four wavefronts and one centre in flight).  Few centres: four wavefronts (the reduction over sixteen is longer, above all
// in double: 3-D, 52 entries of 3019 centres 8.0 / 10.3 us).
constexpr int kSampleBlock = 1024;
template <typename T, int D> constexpr int kSampleFew = sizeof(T) == 4 ? 2048 : D == 2 ? 4096 : 12288;

template <typename T, int D, int BLOCK>
__global__ __launch_bounds__(BLOCK) void sampling_positions_kernel(const T* __restrict__ mixture, T* __restrict__ u,
                                                                   int centres, size_t samples, int chunks) {
    constexpr int G = 1 + D + D * D;
    constexpr int kFlight = BLOCK == kSampleBlock ? 8 : 1;
    __shared__ T red[2 * D][BLOCK / kWave];
    const int b = blockIdx.x / chunks, chunk = blockIdx.x - b * chunks;
    const T* mix_b = mixture + size_t(b) * centres * G;
    T lo[D], hi[D];
    for (int d = 0; d < D; ++d) { lo[d] = T(INFINITY); hi[d] = T(-INFINITY); }
    for (int i = threadIdx.x; i < centres; i += kFlight * BLOCK) {
        T v[kFlight][D];
#pragma unroll
        for (int k = 0; k < kFlight; ++k) {
            const int at = i + k * BLOCK < centres ? i + k * BLOCK : i;
#pragma unroll
            for (int d = 0; d < D; ++d) v[k][d] = mix_b[size_t(at) * G + 1 + d];
        }
#pragma unroll
        for (int k = 0; k < kFlight; ++k)
#pragma unroll
            for (int d = 0; d < D; ++d) {
                lo[d] = v[k][d] < lo[d] ? v[k][d] : lo[d];
                hi[d] = v[k][d] > hi[d] ? v[k][d] : hi[d];
            }
    }
    const int wave = threadIdx.x >> 6;
#pragma unroll
    for (int d = 0; d < D; ++d) {
        for (int off = 1; off < kWave; off <<= 1) {
            const T l2 = __shfl_xor(lo[d], off, kWave), h2 = __shfl_xor(hi[d], off, kWave);
            lo[d] = l2 < lo[d] ? l2 : lo[d];
            hi[d] = h2 > hi[d] ? h2 : hi[d];
        }
        if ((threadIdx.x & 63) == 0) { red[d][wave] = lo[d]; red[D + d][wave] = hi[d]; }
    }
    __syncthreads();
#pragma unroll
    for (int d = 0; d < D; ++d)
#pragma unroll 4        // (all sixteen at once spilled 340 bytes a lane in double: 26 us where the kernel takes 6)
        for (int w = 0; w < BLOCK / kWave; ++w) {
            lo[d] = red[d][w] < lo[d] ? red[d][w] : lo[d];
            hi[d] = red[D + d][w] > hi[d] ? red[D + d][w] : hi[d];
        }
    T* u_b = u + size_t(b) * samples * D;
    const size_t n = samples * D, per = (n + chunks - 1) / chunks;
    const size_t begin = per * chunk, end = begin + per < n ? begin + per : n;
    for (size_t i = begin + threadIdx.x; i < end; i += BLOCK) {
        const int d = int(i % D);
        T l = lo[0], h = hi[0];
#pragma unroll
        for (int k = 1; k < D; ++k) { l = d == k ? lo[k] : l; h = d == k ? hi[k] : h; }
        T v = u_b[i];
        if (D == 2) v = v * T(1.3) - T(0.15);
        u_b[i] = v * (h - l) + l;
    }
}

// Element-wise part of the gradient of one fixed-point iteration (src/gmc/fitting.py:296-311), which sits between the
// evaluations: x1 = x0 (b + 0.05) / c with x0 = |w| + 0.1, b = relu(v + constant) - relu(constant) and
// c = current + 0.05.  As torch operations these were about forty launches over [B][L][N] values (0.2 ms of a layer's
// backward pass, all of it launch latency).
//   prepare: the upstream gradients of both evaluations, d_v = d_b [v + constant > 0] with d_b = d_x1 x0 / c and
//            d_current = -d_x1 x0 ((b + 0.05) / c) / c, and the gradient of the constant, one workgroup per mixture;
//   finish:  grad_out + [sign(w) (d_x1 (b + 0.05) / c + g_weight), sum of the centres' gradients, covariance gradient].
template <typename T, int D>
__global__ __launch_bounds__(kBlock) void relu_fit_prepare_kernel(const T* __restrict__ grad_out, const T* __restrict__ fit,
                                                                  const T* __restrict__ goal, const T* __restrict__ current,
                                                                  const T* __restrict__ constant, T* __restrict__ d_v,
                                                                  T* __restrict__ d_current, T* __restrict__ grad_constant, int N) {
    constexpr int G = 1 + D + D * D;
    __shared__ double wave_sums[kBlock / kWave];
    const T c0 = constant[blockIdx.x];
    const T relu_c = c0 > T(0) ? c0 : (c0 == c0 ? T(0) : c0);
    double acc = 0.0;
    for (int n = threadIdx.x; n < N; n += kBlock) {
        const size_t at = size_t(blockIdx.x) * N + n;
        const T w = fit[at * G], d_x1 = grad_out[at * G], b = goal[at];
        const T x0 = fabs(w) + T(0.1), c = current[at] + T(0.05);
        const T d_b = d_x1 * x0 / c;
        const bool lifted = b + relu_c > T(0);
        d_v[at] = d_b * T(lifted);                       // (a NaN stays one)
        d_current[at] = -d_x1 * x0 * ((b + T(0.05)) / c) / c;
        acc += double(d_b * (T(lifted) - T(c0 > T(0))));
    }
    if (!grad_constant) return;
    acc = wave_sum_to_lane63(acc);
    if ((threadIdx.x & 63) == 63) wave_sums[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) grad_constant[blockIdx.x] = T((wave_sums[0] + wave_sums[1]) + (wave_sums[2] + wave_sums[3]));
}

template <typename T, int D>
__global__ __launch_bounds__(kBlock) void relu_fit_finish_kernel(const T* __restrict__ grad_out, const T* __restrict__ fit,
                                                                 const T* __restrict__ goal, const T* __restrict__ current,
                                                                 const T* __restrict__ g_abs, const T* __restrict__ g_centres,
                                                                 const T* __restrict__ g_centres2, T* __restrict__ grad_fit, size_t n) {
    constexpr int G = 1 + D + D * D;
    const size_t i = size_t(blockIdx.x) * kBlock + threadIdx.x;
    if (i >= n) return;
    const T* go = grad_out + i * G;
    const T* ga = g_abs + i * G;
    T* o = grad_fit + i * G;
    const T w = fit[i * G];
    const T sign = w > T(0) ? T(1) : (w < T(0) ? T(-1) : w);
    o[0] = sign * (go[0] * ((goal[i] + T(0.05)) / (current[i] + T(0.05))) + ga[0]);
#pragma unroll
    for (int d = 0; d < D; ++d) o[1 + d] = go[1 + d] + ((ga[1 + d] + g_centres[i * D + d]) + g_centres2[i * D + d]);
#pragma unroll
    for (int k = 1 + D; k < G; ++k) o[k] = go[k] + ga[k];
}

// The fitting mixture with the iteration's weights in front of it (|w| + 0.1) and, packed, its centres.
template <typename T, int D>
__global__ __launch_bounds__(kBlock) void relu_fit_start_kernel(const T* __restrict__ fit, T* __restrict__ fit_abs,
                                                                T* __restrict__ centres, size_t n) {
    constexpr int G = 1 + D + D * D;
    const size_t i = size_t(blockIdx.x) * kBlock + threadIdx.x;
    if (i >= n) return;
    fit_abs[i * G] = fabs(fit[i * G]) + T(0.1);
#pragma unroll
    for (int k = 1; k < G; ++k) fit_abs[i * G + k] = fit[i * G + k];
#pragma unroll
    for (int d = 0; d < D; ++d) centres[i * D + d] = fit[i * G + 1 + d];
}

// BatchNorm's scaling of the weights (src/gmc/modules.py:417-421): out = mixture with every weight times the factor of its
// (batch entry and) channel, and its gradients.  One pass over the mixture each, bound by HBM: a workgroup walks over a
// chunk of one mixture's scalars, so that the factor is uniform, VEC scalars at a time.  (As torch operations -- slice,
// product, concatenation, and their gradients through zero-filled copies -- the 229 MB of a layer's convolved mixtures
// were read or written about fifteen times: 0.9 ms of a training step, now 0.18 ms.)
// scale [scale_batches][L], scale_batches 1 or B.
template <typename T, int VEC> struct __align__(sizeof(T) * VEC) Scalars { T v[VEC]; };

template <typename T, int D, int VEC>
__global__ __launch_bounds__(kBlock) void scale_weights_kernel(const T* __restrict__ mixture, const T* __restrict__ scale,
                                                               T* __restrict__ out, int L, size_t scalars, int chunks,
                                                               size_t per_chunk, int scale_batches) {
    constexpr unsigned G = 1 + D + D * D;
    const int bl = blockIdx.x / chunks, chunk = blockIdx.x - bl * chunks;
    const T f = scale[scale_batches == 1 ? bl % L : bl];
    const size_t begin = per_chunk * chunk, end = begin + per_chunk < scalars ? begin + per_chunk : scalars;
    const T* __restrict__ in = mixture + size_t(bl) * scalars;
    T* __restrict__ to = out + size_t(bl) * scalars;
    for (size_t i = begin + threadIdx.x * VEC; i < end; i += kBlock * VEC) {
        Scalars<T, VEC> q = *reinterpret_cast<const Scalars<T, VEC>*>(in + i);
        const unsigned r = unsigned(i % G);
#pragma unroll
        for (unsigned k = 0; k < VEC; ++k)
            if (r + k == 0 || r + k == G) q.v[k] *= f;                   // (VEC < G: at most one weight)
        *reinterpret_cast<Scalars<T, VEC>*>(to + i) = q;
    }
}

// grad_mixture = grad_out with every weight's gradient times the factor; partial[bl][chunk] = sum of grad_out times
// mixture over the weights of the chunk (in double; the caller adds them up).  Either result may be absent.
template <typename T, int D, int VEC>
__global__ __launch_bounds__(kBlock) void scale_weights_bwd_kernel(const T* __restrict__ grad_out, const T* __restrict__ mixture,
                                                                   const T* __restrict__ scale, T* __restrict__ grad_mixture,
                                                                   double* __restrict__ partial, int L, size_t scalars, int chunks,
                                                                   size_t per_chunk, int scale_batches) {
    constexpr unsigned G = 1 + D + D * D;
    __shared__ double wave_sums[kBlock / kWave];
    const int bl = blockIdx.x / chunks, chunk = blockIdx.x - bl * chunks;
    const T f = scale[scale_batches == 1 ? bl % L : bl];
    const size_t begin = per_chunk * chunk, end = begin + per_chunk < scalars ? begin + per_chunk : scalars;
    const T* __restrict__ in = grad_out + size_t(bl) * scalars;
    const T* __restrict__ mix = mixture + size_t(bl) * scalars;
    double acc = 0.0;
    for (size_t i = begin + threadIdx.x * VEC; i < end; i += kBlock * VEC) {
        Scalars<T, VEC> q = *reinterpret_cast<const Scalars<T, VEC>*>(in + i);
        const unsigned r = unsigned(i % G);
#pragma unroll
        for (unsigned k = 0; k < VEC; ++k)
            if (r + k == 0 || r + k == G) {
                if (partial) acc = __builtin_fma(double(q.v[k]), double(mix[i + k]), acc);
                q.v[k] *= f;
            }
        if (grad_mixture) *reinterpret_cast<Scalars<T, VEC>*>(grad_mixture + size_t(bl) * scalars + i) = q;
    }
    if (!partial) return;
    acc = wave_sum_to_lane63(acc);
    if ((threadIdx.x & 63) == 63) wave_sums[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = (wave_sums[0] + wave_sums[1]) + (wave_sums[2] + wave_sums[3]);
}

// Workgroups per mixture: about 4096 in all, each with at least 16 scalars per lane.  A chunk is a whole number of
// vectors for every VEC.
static int scale_weights_chunks(const gmc_shape& s) {
    const size_t BL = size_t(s.B) * s.L, scalars = size_t(s.M) * (1 + s.D + s.D * s.D);
    size_t chunks = BL > 0 ? (4096 + BL - 1) / BL : 1;
    const size_t most = scalars / (16 * kBlock);
    if (chunks > most) chunks = most;
    return int(chunks < 1 ? 1 : chunks);
}

// flags |= 1: a NaN or an infinity; |= 2: a matrix with determinant <= 0 (util/mixture.h:85-93)
template <typename T, int D>
__global__ __launch_bounds__(kBlock) void validate_kernel(const T* __restrict__ mixture, size_t n, int* __restrict__ flags) {
    constexpr int G = 1 + D + D * D;
    const size_t i = size_t(blockIdx.x) * kBlock + threadIdx.x;
    int bad = 0;
    if (i < n) {
        const T* g = mixture + i * G;
        bool finite = true;
#pragma unroll
        for (int k = 0; k < G; ++k) finite = finite & (fabs(double(g[k])) <= 1.7976931348623157e308);   // false for NaN and inf
        const T* c = g + 1 + D;
        double det;
        if constexpr (D == 2) det = double(c[0]) * c[3] - double(c[1]) * c[2];
        else det = double(c[0]) * (double(c[4]) * c[8] - double(c[5]) * c[7]) - double(c[1]) * (double(c[3]) * c[8] - double(c[5]) * c[6]) +
                   double(c[2]) * (double(c[3]) * c[7] - double(c[4]) * c[6]);
        bad = (finite ? 0 : 1) | (det > 0.0 ? 0 : 2);
    }
    if (__ballot(bad != 0) != 0ull && bad) atomicOr(flags, bad);
}

}  // namespace gmc

using gmc::EpiArgs;

template <int KIND>
static int consumer_dispatch(const void* mixture, const void* points, size_t mixture_stride, int point_stride,
                             const void* constant, const void* goal, const void* weights, void* out, double* moments,
                             const gmc_shape& s, hipStream_t st) {
#define GMC_GO(T, DD) do { EpiArgs<T> e{(const T*)constant, (const T*)goal, (const T*)weights, (T*)out, moments}; \
        return gmc::launch_consumer<T, DD, KIND>((const T*)mixture, (const T*)points, mixture_stride, point_stride, e, s.B, s.L, s.M, s.N, st); } while (0)
    if (s.dtype == GMC_F32) { if (s.D == 2) GMC_GO(float, 2); else GMC_GO(float, 3); }
    else { if (s.D == 2) GMC_GO(double, 2); else GMC_GO(double, 3); }
#undef GMC_GO
}

extern "C" {

static int consumer_shape(const gmc_shape* shape) {
    const int rc = gmc::check_shape(shape);
    if (rc != GMC_OK) return rc;
    if (shape->Bx != shape->B || shape->Lx != shape->L) return GMC_E_SHAPE;      // one set of points per mixture
    return GMC_OK;
}

int gmc_relu_fit_goal(const void* target_mixture, const void* constant, const void* fitting_mixture, void* goal,
                      const gmc_shape* shape, void* stream) {
    const int rc = consumer_shape(shape);
    if (rc != GMC_OK) return rc;
    if (size_t(shape->B) * shape->L * shape->N == 0) return GMC_OK;
    if (!constant || !fitting_mixture || !goal || (!target_mixture && shape->M > 0)) return GMC_E_NULL;
    const int G = 1 + shape->D + shape->D * shape->D;
    const size_t elt = shape->dtype == GMC_F32 ? 4 : 8;
    const void* centres = (const char*)fitting_mixture + elt;                      // first position of the first Gaussian
    return consumer_dispatch<gmc::kEpiReluShift>(target_mixture, centres, size_t(shape->N) * G, G, constant, nullptr, nullptr,
                                                  goal, nullptr, *shape, (hipStream_t)stream);
}

int gmc_relu_fit_step(const void* fitting_mixture, const void* x_in, const void* goal, void* x_out, const gmc_shape* shape,
                      void* stream) {
    const int rc = consumer_shape(shape);
    if (rc != GMC_OK) return rc;
    if (shape->M != shape->N) return GMC_E_SHAPE;                                  // the points are the mixture's own centres
    if (size_t(shape->B) * shape->L * shape->N == 0) return GMC_OK;
    if (!fitting_mixture || !x_in || !goal || !x_out) return GMC_E_NULL;
    if (x_in == x_out) return GMC_E_SHAPE;                                         // every workgroup reads all of x_in
    const int G = 1 + shape->D + shape->D * shape->D;
    const size_t elt = shape->dtype == GMC_F32 ? 4 : 8;
    const void* centres = (const char*)fitting_mixture + elt;
    return consumer_dispatch<gmc::kEpiRatio>(fitting_mixture, centres, size_t(shape->N) * G, G, nullptr, goal, x_in, x_out,
                                              nullptr, *shape, (hipStream_t)stream);
}

size_t gmc_eval_cov_moments_bytes(const gmc_shape* shape) {
    if (consumer_shape(shape) != GMC_OK) return 0;
    return size_t(shape->B) * shape->L * gmc::consumer_chunks(shape->N) * 3 * sizeof(double);
}

int gmc_eval_cov_moments(const void* mixture, const void* constant, const void* xes, double* moments, size_t moments_bytes,
                         void* sd, void* mean, void* inv_sd, void* running_sd, void* running_mean, double alpha,
                         const gmc_shape* shape, int per_sample, void* stream) {
    const int rc = consumer_shape(shape);
    if (rc != GMC_OK) return rc;
    const int slots = per_sample ? shape->B * shape->L : shape->L;
    if (slots == 0) return GMC_OK;
    if (!sd || !mean) return GMC_E_NULL;
    if ((running_sd == nullptr) != (running_mean == nullptr)) return GMC_E_NULL;
    hipStream_t st = (hipStream_t)stream;
    const bool any = size_t(shape->B) * shape->N > 0;
    if (any) {
        if (!moments) return GMC_E_NULL;
        if (moments_bytes < gmc_eval_cov_moments_bytes(shape)) return GMC_E_WORKSPACE;
        if (!constant || !xes || (!mixture && shape->M > 0)) return GMC_E_NULL;
        const int r2 = consumer_dispatch<gmc::kEpiMoments>(mixture, xes, size_t(shape->N) * shape->D, shape->D, constant, nullptr,
                                                            nullptr, nullptr, moments, *shape, st);
        if (r2 != GMC_OK) return r2;
    }
    // no values at all: no record is read, and the statistics are undefined (NaN), as torch.std_mean of nothing
    const int B = any ? shape->B : 0, chunks = any ? gmc::consumer_chunks(shape->N) : 0;
    const dim3 grid(unsigned((slots + gmc::kBlock / gmc::kWave - 1) / (gmc::kBlock / gmc::kWave)));
    if (shape->dtype == GMC_F32)
        gmc::moments_finish_kernel<float><<<grid, dim3(gmc::kBlock), 0, st>>>(moments, (float*)sd, (float*)mean, (float*)inv_sd,
                                                                              (float*)running_sd, (float*)running_mean, alpha, slots,
                                                                              B, shape->L, chunks, per_sample);
    else
        gmc::moments_finish_kernel<double><<<grid, dim3(gmc::kBlock), 0, st>>>(moments, (double*)sd, (double*)mean, (double*)inv_sd,
                                                                               (double*)running_sd, (double*)running_mean, alpha, slots,
                                                                               B, shape->L, chunks, per_sample);
    return hipGetLastError() == hipSuccess ? GMC_OK : GMC_E_LAUNCH;
}

int gmc_batch_norm_sampling_positions(const void* mixture, void* uniform_in_positions_out, const gmc_shape* shape, void* stream) {
    const int rc = consumer_shape(shape);
    if (rc != GMC_OK) return rc;
    const size_t samples = size_t(shape->L) * shape->N;
    if (shape->B == 0 || samples == 0) return GMC_OK;
    if (!uniform_in_positions_out || (!mixture && shape->M > 0)) return GMC_E_NULL;
    const int centres = shape->L * shape->M;
    hipStream_t st = (hipStream_t)stream;
    // a workgroup per 16384 numbers, at most 64 per batch entry (each reads all centres of its entry)
    const size_t wanted = (samples * shape->D + 16383) / 16384;
    const int chunks = int(wanted < 1 ? 1 : (wanted > 64 ? 64 : wanted));
    const dim3 grid{unsigned(shape->B) * unsigned(chunks)};
#define GMC_SPB(T, DD, BLOCK) gmc::sampling_positions_kernel<T, DD, BLOCK><<<grid, dim3(BLOCK), 0, st>>>((const T*)mixture, (T*)uniform_in_positions_out, centres, samples, chunks)
#define GMC_SP(T, DD) do { if (centres <= gmc::kSampleFew<T, DD>) GMC_SPB(T, DD, gmc::kBlock); else GMC_SPB(T, DD, gmc::kSampleBlock); } while (0)
    if (shape->dtype == GMC_F32) { if (shape->D == 2) GMC_SP(float, 2); else GMC_SP(float, 3); }
    else { if (shape->D == 2) GMC_SP(double, 2); else GMC_SP(double, 3); }
#undef GMC_SP
#undef GMC_SPB
    return hipGetLastError() == hipSuccess ? GMC_OK : GMC_E_LAUNCH;
}

#define GMC_FIT(KERNEL, GRID, ...) do { \
        const dim3 grid{unsigned(GRID)}, block{gmc::kBlock}; \
        if (shape->dtype == GMC_F32) { using T = float; if (shape->D == 2) gmc::KERNEL<T, 2><<<grid, block, 0, st>>>(__VA_ARGS__); else gmc::KERNEL<T, 3><<<grid, block, 0, st>>>(__VA_ARGS__); } \
        else { using T = double; if (shape->D == 2) gmc::KERNEL<T, 2><<<grid, block, 0, st>>>(__VA_ARGS__); else gmc::KERNEL<T, 3><<<grid, block, 0, st>>>(__VA_ARGS__); } \
        return hipGetLastError() == hipSuccess ? GMC_OK : GMC_E_LAUNCH; } while (0)

int gmc_relu_fit_grad_start(const void* fitting_mixture, void* fitting_abs, void* centres, const gmc_shape* shape, void* stream) {
    const int rc = consumer_shape(shape);
    if (rc != GMC_OK) return rc;
    const size_t n = size_t(shape->B) * shape->L * shape->N;
    if (n == 0) return GMC_OK;
    if (!fitting_mixture || !fitting_abs || !centres) return GMC_E_NULL;
    hipStream_t st = (hipStream_t)stream;
    GMC_FIT(relu_fit_start_kernel, (n + gmc::kBlock - 1) / gmc::kBlock, (const T*)fitting_mixture, (T*)fitting_abs, (T*)centres, n);
}

int gmc_relu_fit_grad_prepare(const void* grad_out, const void* fitting_mixture, const void* goal, const void* current,
                              const void* constant, void* d_value, void* d_current, void* grad_constant, const gmc_shape* shape,
                              void* stream) {
    const int rc = consumer_shape(shape);
    if (rc != GMC_OK) return rc;
    const size_t BL = size_t(shape->B) * shape->L;
    if (BL == 0) return GMC_OK;
    if (!constant || (shape->N > 0 && (!grad_out || !fitting_mixture || !goal || !current || !d_value || !d_current))) return GMC_E_NULL;
    hipStream_t st = (hipStream_t)stream;
    GMC_FIT(relu_fit_prepare_kernel, BL, (const T*)grad_out, (const T*)fitting_mixture, (const T*)goal, (const T*)current,
            (const T*)constant, (T*)d_value, (T*)d_current, (T*)grad_constant, shape->N);
}

int gmc_relu_fit_grad_finish(const void* grad_out, const void* fitting_mixture, const void* goal, const void* current,
                             const void* grad_abs, const void* grad_centres, const void* grad_centres2, void* grad_fitting,
                             const gmc_shape* shape, void* stream) {
    const int rc = consumer_shape(shape);
    if (rc != GMC_OK) return rc;
    const size_t n = size_t(shape->B) * shape->L * shape->N;
    if (n == 0) return GMC_OK;
    if (!grad_out || !fitting_mixture || !goal || !current || !grad_abs || !grad_centres || !grad_centres2 || !grad_fitting) return GMC_E_NULL;
    hipStream_t st = (hipStream_t)stream;
    GMC_FIT(relu_fit_finish_kernel, (n + gmc::kBlock - 1) / gmc::kBlock, (const T*)grad_out, (const T*)fitting_mixture, (const T*)goal,
            (const T*)current, (const T*)grad_abs, (const T*)grad_centres, (const T*)grad_centres2, (T*)grad_fitting, n);
}
#undef GMC_FIT

size_t gmc_scale_weights_chunks(const gmc_shape* shape) {
    return consumer_shape(shape) == GMC_OK ? size_t(gmc::scale_weights_chunks(*shape)) : 0;
}

static bool aligned16(const void* a, const void* b) { return ((uintptr_t(a) | uintptr_t(b)) & 15) == 0; }

int gmc_scale_weights(const void* mixture, const void* scale, void* out, const gmc_shape* shape, int scale_per_batch, void* stream) {
    const int rc = consumer_shape(shape);
    if (rc != GMC_OK) return rc;
    const size_t BL = size_t(shape->B) * shape->L, scalars = size_t(shape->M) * (1 + shape->D + shape->D * shape->D);
    if (BL * scalars == 0) return GMC_OK;
    if (!mixture || !scale || !out) return GMC_E_NULL;
    const int chunks = gmc::scale_weights_chunks(*shape);
    const size_t per = ((scalars + chunks - 1) / chunks + 3) / 4 * 4;
    const int batches = scale_per_batch ? shape->B : 1;
    const dim3 grid(unsigned(BL * chunks)), block(gmc::kBlock);
    hipStream_t st = (hipStream_t)stream;
#define GMC_SW(T, DD, V) gmc::scale_weights_kernel<T, DD, V><<<grid, block, 0, st>>>((const T*)mixture, (const T*)scale, (T*)out, shape->L, scalars, chunks, per, batches)
    // 16-byte accesses where every mixture starts at a multiple of 16 bytes
    const bool f32 = shape->dtype == GMC_F32;
    const bool wide = aligned16(mixture, out) && scalars % (f32 ? 4 : 2) == 0;
    if (f32) {
        if (shape->D == 2) { if (wide) GMC_SW(float, 2, 4); else GMC_SW(float, 2, 1); }
        else { if (wide) GMC_SW(float, 3, 4); else GMC_SW(float, 3, 1); }
    } else {
        if (shape->D == 2) { if (wide) GMC_SW(double, 2, 2); else GMC_SW(double, 2, 1); }
        else { if (wide) GMC_SW(double, 3, 2); else GMC_SW(double, 3, 1); }
    }
#undef GMC_SW
    return hipGetLastError() == hipSuccess ? GMC_OK : GMC_E_LAUNCH;
}

int gmc_scale_weights_bwd(const void* grad_out, const void* mixture, const void* scale, void* grad_mixture, double* partial,
                          const gmc_shape* shape, int scale_per_batch, void* stream) {
    const int rc = consumer_shape(shape);
    if (rc != GMC_OK) return rc;
    const size_t BL = size_t(shape->B) * shape->L, scalars = size_t(shape->M) * (1 + shape->D + shape->D * shape->D);
    if (!grad_mixture && !partial) return GMC_OK;
    const int chunks = gmc::scale_weights_chunks(*shape);
    hipStream_t st = (hipStream_t)stream;
    if (BL * scalars == 0) {
        if (partial && BL > 0) gmc::zero_async(partial, BL * chunks, st);
        return hipGetLastError() == hipSuccess ? GMC_OK : GMC_E_LAUNCH;
    }
    if (!grad_out || !scale || (partial && !mixture)) return GMC_E_NULL;
    const size_t per = ((scalars + chunks - 1) / chunks + 3) / 4 * 4;
    const int batches = scale_per_batch ? shape->B : 1;
    const dim3 grid(unsigned(BL * chunks)), block(gmc::kBlock);
#define GMC_SW(T, DD, V) gmc::scale_weights_bwd_kernel<T, DD, V><<<grid, block, 0, st>>>((const T*)grad_out, (const T*)mixture, (const T*)scale, (T*)grad_mixture, partial, shape->L, scalars, chunks, per, batches)
    const bool f32 = shape->dtype == GMC_F32;
    const bool wide = aligned16(grad_out, grad_mixture) && scalars % (f32 ? 4 : 2) == 0;
    if (f32) {
        if (shape->D == 2) { if (wide) GMC_SW(float, 2, 4); else GMC_SW(float, 2, 1); }
        else { if (wide) GMC_SW(float, 3, 4); else GMC_SW(float, 3, 1); }
    } else {
        if (shape->D == 2) { if (wide) GMC_SW(double, 2, 2); else GMC_SW(double, 2, 1); }
        else { if (wide) GMC_SW(double, 3, 2); else GMC_SW(double, 3, 1); }
    }
#undef GMC_SW
    return hipGetLastError() == hipSuccess ? GMC_OK : GMC_E_LAUNCH;
}

int gmc_validate_mixture(const void* mixture, int32_t* flags, const gmc_shape* shape, void* stream) {
    const int rc = gmc::check_shape(shape);
    if (rc != GMC_OK) return rc;
    if (!flags) return GMC_E_NULL;
    hipStream_t st = (hipStream_t)stream;
    gmc::zero_async(flags, 1, st);
    const size_t n = size_t(shape->B) * shape->L * shape->M;
    if (n > 0) {
        if (!mixture) return GMC_E_NULL;
        const dim3 grid(unsigned((n + gmc::kBlock - 1) / gmc::kBlock));
#define GMC_VAL(T, DD) gmc::validate_kernel<T, DD><<<grid, dim3(gmc::kBlock), 0, st>>>((const T*)mixture, n, flags)
        if (shape->dtype == GMC_F32) { if (shape->D == 2) GMC_VAL(float, 2); else GMC_VAL(float, 3); }
        else { if (shape->D == 2) GMC_VAL(double, 2); else GMC_VAL(double, 3); }
#undef GMC_VAL
    }
    return hipGetLastError() == hipSuccess ? GMC_OK : GMC_E_LAUNCH;
}

}  // extern "C"
