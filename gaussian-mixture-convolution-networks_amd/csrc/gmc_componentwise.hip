// Component-wise evaluation: values[b,l,n,m] = w_m * N(x_n; b_m, C_m) without the sum over components
// (the pure-torch evaluate_componentwise_inversed of the reference, src/gmc/mixture.py:152-180, used by its
// fitting code).  The output has one scalar per pair, so the kernels are bound by HBM stores (forward) and loads
// (backward), not by the vector ALU: lanes own Gaussians (the fastest output dimension, coalesced stores), the
// points of a workgroup's chunk are wave-uniform and arrive through scalar loads.
#include "gmc_common.h"

namespace gmc {

int check_shape(const gmc_shape* s);

constexpr int kCwPoints = 64;      // points per workgroup
template <typename T, int Q> struct __align__(sizeof(T) * Q) CwVec { T v[Q]; };

template <typename T, int D>
__global__ __launch_bounds__(kBlock) void componentwise_fwd_kernel(const T* __restrict__ mixture, const T* __restrict__ xes,
                                                                  T* __restrict__ out, int L, int M, int N, int Bx, int Lx,
                                                                  int m_tiles, int first_mixture, int chunks, bool covariance_form) {
    constexpr int G = 1 + D + D * D;
    const T* exp2_tab = exp2_table<T>();
    if constexpr (sizeof(T) == 8) __syncthreads();          // the table is complete (all wavefronts are still here)
    int id = blockIdx.x;
    const int chunk = id % chunks; id /= chunks;
    const int tile = id % m_tiles;
    const int bl = first_mixture + id / m_tiles;
    const int b = bl / L, l = bl - b * L;
    const int xb = b < Bx ? b : Bx - 1, xl = l < Lx ? l : Lx - 1;
    // A wavefront owns one slice of 64 Gaussians; with fewer than four slices in this tile the four wavefronts share
    // the points of the chunk instead of idling (see the backward kernel).
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;    // wave-uniform for the compiler too
    const int slices_total = (M + kWave - 1) / kWave;
    const int slices_here = slices_total - tile * 4 < 4 ? slices_total - tile * 4 : 4;
    const int reps = 4 / slices_here;
    const int slice = wave % slices_here, rep = wave / slices_here;
    if (rep >= reps) return;
    const int m = (tile * 4 + slice) * kWave + lane;
    const bool valid = m < M;
    const T* __restrict__ x_bl = xes + (size_t(xb) * Lx + xl) * N * D;
    T r[Rec<T, D>::kStride];
    {
        const Derived<D> dv = derive<T, D>(mixture + (size_t(bl) * M + (valid ? m : 0)) * G, covariance_form);
        store_record<T, D>(r, dv, true, dv.w * dv.norm, 0);
    }
    const int per_rep = (kCwPoints + reps - 1) / reps;
    const int n_begin = chunk * kCwPoints + rep * per_rep;
    int n_end = n_begin + per_rep < (chunk + 1) * kCwPoints ? n_begin + per_rep : (chunk + 1) * kCwPoints;
    n_end = n_end < N ? n_end : N;
    for (int n = n_begin; n < n_end; ++n) {
        T x[D];
#pragma unroll
        for (int d = 0; d < D; ++d) x[d] = x_bl[size_t(n) * D + d];
        T y[D];
        const T q = quad_form<T, D, true>(r, x, y);
        if (valid) out[(size_t(bl) * N + n) * M + m] = r[Rec<T, D>::kAmp] * pair_exp2(-q, exp2_tab);
    }
}

// The same with four Gaussians per lane (float32): a power of two of lanes holds a point's row, the others of a wavefront the
// following points, so that few Gaussians leave no lanes idle.  WIDE, where every row starts at a multiple of 16 bytes: a
// lane's Gaussians are neighbours and its values leave with one store; elsewhere they lie a row of lanes apart.  The workgroup
// prepares the tile's Gaussians once, through LDS, and walks over `points_per_chunk` points; four steps of a wavefront are in
// flight.  Taken (cw_wide_forward) for at most 64 Gaussians (32 without WIDE), where the kernel above leaves lanes or
// wavefronts idle, and for launches of fewer than 512 of its workgroups; with more of both it takes between 0.8 and 1.3 of the
// time, and in double, where a lane prepares two, small calls take up to 1.4 times as long.  Kernel above / this one, us: 1600 x
// 16 Gaussians at 1000 points, 2-D, 65 / 20;  800 x 44 at 900, 3-D, 45 / 28;  320 x 32 at 4096 57 / 30 (167 MB of values,
// 5.6 TB/s: bound by the stores);  1 x 300 at 3000, 3-D, 11.9 / 4.8;  1 x 32 at 784 3.8 / 2.6.  Over 11000 drawn calls the
// median is 0.71 of the time, none slower.
template <int D, bool WIDE>
__global__ __launch_bounds__(kBlock) void componentwise_fwd_wide_kernel(const float* __restrict__ mixture, const float* __restrict__ xes,
                                                                       float* __restrict__ out, int L, int M, int N, int Bx, int Lx,
                                                                       int m_tiles, int first_mixture, int chunks,
                                                                       int points_per_chunk, bool covariance_form) {
    constexpr int G = 1 + D + D * D, S = Rec<float, D>::kStride, Q = 4, kTileG = kWave * Q, U = 4;
    __shared__ __attribute__((aligned(16))) float lds[kTileG * S];
    int id = blockIdx.x;
    const int chunk = id % chunks; id /= chunks;
    const int tile = id % m_tiles;
    const int bl = first_mixture + id / m_tiles;
    const int b = bl / L, l = bl - b * L;
    const int xb = b < Bx ? b : Bx - 1, xl = l < Lx ? l : Lx - 1;
    const float* __restrict__ x_bl = xes + (size_t(xb) * Lx + xl) * N * D;
    const int here = M - tile * kTileG < kTileG ? M - tile * kTileG : kTileG;
    if (int(threadIdx.x) < here) {
        const Derived<D> dv = derive<float, D>(mixture + (size_t(bl) * M + tile * kTileG + threadIdx.x) * G, covariance_form);
        store_record<float, D>(lds + threadIdx.x * S, dv, true, dv.w * dv.norm, 0);
    }
    __syncthreads();
    int shift = 6;                                          // log2 of the lanes of a row
    while (shift > 0 && (Q << (shift - 1)) >= here) --shift;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int slot = lane & ((1 << shift) - 1), rows = 64 >> shift;
    // Gaussian q of this lane
    const int first = WIDE ? slot * Q : slot, apart = WIDE ? 1 : 1 << shift;
    const bool active = first < here;
    float r[Q][Rec<float, D>::kUsed];
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int i = 0; i < Rec<float, D>::kUsed; ++i) r[q][i] = lds[(first + q * apart < here ? first + q * apart : 0) * S + i];
    const int n_first = chunk * points_per_chunk;
    const int n_end = n_first + points_per_chunk < N ? n_first + points_per_chunk : N;
    float* __restrict__ to = out + size_t(bl) * N * M + tile * kTileG + first;
    for (int n0 = n_first + wave * rows + (lane >> shift); n0 - (lane >> shift) < n_end; n0 += 4 * rows * U) {
        float x[U][D];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int n = n0 + u * 4 * rows < n_end ? n0 + u * 4 * rows : n_end - 1;
#pragma unroll
            for (int d = 0; d < D; ++d) x[u][d] = x_bl[size_t(n) * D + d];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int n = n0 + u * 4 * rows;
            float f[Q], e[Q];
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                float y[D];
                f[q] = quad_form<float, D, true>(r[q], x[u], y);
            }
            pair_exp2_batch(f, e);
            if (active && n < n_end) {
                if constexpr (WIDE) {
                    CwVec<float, Q> v;
#pragma unroll
                    for (int q = 0; q < Q; ++q) v.v[q] = r[q][Rec<float, D>::kAmp] * e[q];
                    *reinterpret_cast<CwVec<float, Q>*>(to + size_t(n) * M) = v;
                } else {
#pragma unroll
                    for (int q = 0; q < Q; ++q)
                        if (first + q * apart < here) to[size_t(n) * M + q * apart] = r[q][Rec<float, D>::kAmp] * e[q];
                }
            }
        }
    }
}

// Layout of the backward pass: the 64 lanes of a wavefront are 4 rows (points) by 16 columns, a column holds Q Gaussians,
// so that the coordinates of a point are fetched once for Q pairs.  Where every row of grad_out starts at a multiple of
// the vector (`wide`), a column's Gaussians lie next to each other and one access per lane fetches the values of 16 Q
// Gaussians at 4 points; elsewhere they lie 16 apart and Q accesses fetch 64 bytes of a row each.  A wavefront owns one
// such slice of Gaussians; with fewer than four slices in its group the four wavefronts of a workgroup share the points of
// the chunk.  (The forward pass, which only stores, is faster with lanes = Gaussians: 800 x 128 Gaussians at 784 points in
// 2-D 74 us against 107 us in this layout.)
constexpr int kCwPointsMax = 1024; // most points per workgroup of the backward pass (the size of its LDS copy of dL/dx)

// Gaussians per lane: one or, in float32, two -- a lane prepares them one after the other and holds a record and sums for
// each.  Two where the mixtures fill their slices (groups of 128 components cover at most a tenth more than groups of 64)
// and the launch has work for the chip (512 pieces of 64 x 64 pairs).  Measured, both gradients, one / two / four a lane in
// us (float32 2-D): 800 x 128 Gaussians at 784 points 107 / 95 / 100, 800 x 132 123 / 147 / 137, 20 x 512 at 4096
// 52 / 47 / 52, 1000 x 16 at 1000 28 / 41 / 73, 64 x 4 at 1 8.7 / 9.8 / 11.5; 3-D: 800 x 128 132 / 122 / -, 1000 x 129 at
// 128 46 / 66 / -; float64 (2-D): 400 x 128 at 784 111 / 111 / -, 1000 x 1200 at 16 161 / 174 / -.
template <typename T> static bool cw_two_per_lane(const gmc_shape& s) {
    if (sizeof(T) == 8) return false;
    const size_t groups = (size_t(s.M) + 63) / 64, pairs_of_groups = (groups + 1) / 2;
    return 20 * pairs_of_groups <= 11 * groups && size_t(s.B) * s.L * groups * ((size_t(s.N) + 63) / 64) >= 512;
}

struct CwSlices { int slice, rep, reps; };

// the share of a wavefront: slice of the Gaussians (of a group of one per wavefront, -1: none) and repetition over the points
__device__ __forceinline__ CwSlices cw_share(int M, int group, int per_slice, int waves, int wave) {
    const int left = (M + per_slice - 1) / per_slice - group * waves;
    const int here = left < waves ? left : waves;
    const int reps = waves / here;
    const int rep = wave / here;
    return CwSlices{rep < reps ? wave % here : -1, rep, reps};
}

// Sums of 4 (or 8) values over the 16 lanes of a DPP row at once: in every step the halves of a group exchange the
// values they do not keep.  Returns, in lane `lane` of the row, the total of value cw_sum_index(lane) (4 values: bits 3
// and 2 of the lane choose; 8 values: bits 3, 2 and 1).
template <typename T, int COUNT>
__device__ __forceinline__ T cw_row_sums(const T (&v)[COUNT], int lane) {
    static_assert(COUNT == 4 || COUNT == 8, "");
    T a[COUNT / 2];
    const bool b3 = (lane & 8) != 0, b2 = (lane & 4) != 0, b1 = (lane & 2) != 0;
#pragma unroll
    for (int i = 0; i < COUNT / 2; ++i) {
        const T low = v[2 * i], high = v[2 * i + 1];
        a[i] = (b3 ? high : low) + dpp_mov<0x128>(b3 ? low : high);         // row_ror:8
    }
    T c[COUNT / 4];
#pragma unroll
    for (int i = 0; i < COUNT / 4; ++i) {
        const T low = a[2 * i], high = a[2 * i + 1];
        c[i] = (b2 ? high : low) + dpp_mov<0x141>(b2 ? low : high);         // row_half_mirror: the other half of eight
    }
    T s;
    if constexpr (COUNT == 8) {
        const T low = c[0], high = c[1];
        s = (b1 ? high : low) + dpp_mov<0x4e>(b1 ? low : high);             // quad_perm 2 3 0 1
    } else {
        s = c[0] + dpp_mov<0x4e>(c[0]);
    }
    return s + dpp_mov<0xb1>(s);                                            // quad_perm 1 0 3 2
}
template <int COUNT> __device__ __forceinline__ int cw_sum_index(int lane) {
    return ((lane >> 3) & 1) + 2 * ((lane >> 2) & 1) + (COUNT == 8 ? 4 * ((lane >> 1) & 1) : 0);
}

// Backward: grad_out [B][L][N][M] weights every pair on its own and is read once.  A row's point meets Q Gaussians per
// lane before its dL/dx is reduced, over the 16 columns only; four points of a row (16 of the wavefront) go through that
// reduction together, and their grad_out values are in flight together.  Per-Gaussian sums stay in the lane's
// registers over the points, are added over the rows and over the wavefronts that share a slice at the end, and leave
// with one atomic per scalar and workgroup; dL/dx of a point goes through the workgroup's LDS copy and leaves with one
// atomic (or, when one workgroup sees all Gaussians of the point, one store) per scalar.  With lanes = Gaussians and every
// point's dL/dx reduced over 64 lanes / now (us, float32, both gradients): 800 x 128 Gaussians at 784 points in 2-D
// 128 / 102 (3.2 TB/s of grad_out), in 3-D 199 / 130; 20 x 512 at 4096 points 118 / 49 and 272 / 66; 1 x 2 mixtures of 4 at
// 2 points 8.3 / 7.9.  At the first shape 31 instructions per 64 pairs take about 45 us of the 102, and grad_out is read at
// 3.3 TB/s where the backward pass of the convolution reads its own at 4.9: not bound by issue, and what holds its reads at
// that rate is not shown (the next rows fetched ahead and batched exponentials change nothing).
constexpr int kCwSteps = 4;        // points of a row per round

template <typename T, int D, int Q, int WAVES, bool NEED_GM, bool NEED_GX>
__global__ __launch_bounds__(WAVES * kWave) __attribute__((amdgpu_waves_per_eu(WAVES > 4 ? 4 : sizeof(T) == 8 ? 2 : D == 3 ? 3 : 4)))
void componentwise_bwd_kernel(const T* __restrict__ grad_out, const T* __restrict__ mixture,
                                                                  const T* __restrict__ xes, T* __restrict__ sums,
                                                                  T* __restrict__ grad_xes, int L, int M, int N, int Bx,
                                                                  int Lx, int m_groups, int first_mixture, int chunks,
                                                                  int points_per_chunk, bool shared_points, bool wide, bool covariance_form) {
    constexpr int G = 1 + D + D * D, U = kCwSteps, kThreads = WAVES * kWave;
    constexpr int NR = 1 + D + D * (D + 1) / 2;
    constexpr int kU = Rec<T, D>::kU;
    __shared__ T point_grad[NEED_GX ? kCwPointsMax * D : 1];
    __shared__ T shared_sums[NEED_GM ? WAVES * 16 * Q * NR : 1];
    const T* exp2_tab = exp2_table<T>();
    if constexpr (sizeof(T) == 8) __syncthreads();          // the table is complete
    int id = blockIdx.x;
    const int chunk = id % chunks; id /= chunks;
    const int group = id % m_groups;
    const int bl = first_mixture + id / m_groups;
    const int b = bl / L, l = bl - b * L;
    const int xb = b < Bx ? b : Bx - 1, xl = l < Lx ? l : Lx - 1;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, row = lane >> 4, col = lane & 15;
    const CwSlices share = cw_share(M, group, 16 * Q, WAVES, wave);
    // Gaussian q of this lane is m0 + q * apart
    const int apart = wide ? 1 : 16;
    const int m0 = (group * WAVES + share.slice) * 16 * Q + (wide ? col * Q : col);
    const size_t x_off = (size_t(xb) * Lx + xl) * N;
    const T* __restrict__ x_bl = xes + x_off * D;
    if (NEED_GX) {
        for (int i = threadIdx.x; i < points_per_chunk * D; i += kThreads) point_grad[i] = T(0);
        __syncthreads();
    }
    const int chunk_begin = chunk * points_per_chunk;
    T rs[Q][NR];
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int i = 0; i < NR; ++i) rs[q][i] = T(0);
    if (share.slice >= 0) {
        T r[Q][Rec<T, D>::kStride], ua[Q][kU];      // ua = -amp * u: dL/dx takes k*y against it
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const Derived<D> dv = derive<T, D>(mixture + (size_t(bl) * M + (m0 + q * apart < M ? m0 + q * apart : 0)) * G, covariance_form);
            // amplitude for dL/dx as in the summed backward kernel: w norm / (0.5 log2 e)
            store_record<T, D>(r[q], dv, true, over_half_log2e<T>(dv.w * dv.norm), 0);
#pragma unroll
            for (int i = 0; i < kU; ++i) ua[q][i] = -r[q][Rec<T, D>::kAmp] * r[q][i];
        }
        const int per_rep = ((points_per_chunk + share.reps - 1) / share.reps + 4 * U - 1) / (4 * U) * (4 * U);
        const int n_begin = chunk_begin + share.rep * per_rep;
        int n_end = n_begin + per_rep < chunk_begin + points_per_chunk ? n_begin + per_rep : chunk_begin + points_per_chunk;
        n_end = n_end < N ? n_end : N;
        const T* __restrict__ go_bl = grad_out + size_t(bl) * N * M;
        // values and coordinates of the row's next U points; beyond the end and beyond M: zeros, which add nothing
        auto fetch = [&](int n0, CwVec<T, Q> (&go)[U], T (&xs)[U][D]) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int at = n0 + u * 4 + row;
                const int n = at < n_end ? at : n_end - 1;
                const T* from = go_bl + size_t(n) * M + m0;
                if (wide && m0 < M) {                       // (M is a multiple of Q)
                    go[u] = *reinterpret_cast<const CwVec<T, Q>*>(from);
                } else {
#pragma unroll
                    for (int q = 0; q < Q; ++q) go[u].v[q] = m0 + q * apart < M ? from[q * apart] : T(0);
                }
#pragma unroll
                for (int d = 0; d < D; ++d) xs[u][d] = x_bl[size_t(n) * D + d];
            }
        };
        for (int n0 = n_begin; n0 < n_end; n0 += 4 * U) {
            CwVec<T, Q> go[U];
            T xs[U][D];
            fetch(n0, go, xs);
            T vs[D][U];                                     // dL/dx of the row's points, this lane's Gaussians
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const bool in = n0 + u * 4 + row < n_end;
                T v[D];
#pragma unroll
                for (int d = 0; d < D; ++d) v[d] = T(0);
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    T y[D];
                    const T e = quad_form<T, D, true>(r[q], xs[u], y);
                    const T k = (in && m0 + q * apart < M) ? pair_exp2(-e, exp2_tab) * go[u].v[q] : T(0);
                    T ky[D];
#pragma unroll
                    for (int d = 0; d < D; ++d) ky[d] = k * y[d];
                    if (NEED_GM) {
                        rs[q][0] += k;
                        int at = 1 + D;
#pragma unroll
                        for (int a = 0; a < D; ++a) {
                            rs[q][1 + a] += ky[a];
#pragma unroll
                            for (int c = a; c < D; ++c) { rs[q][at] = fma_(ky[a], y[c], rs[q][at]); ++at; }
                        }
                    }
                    if (NEED_GX) {
                        // -(amp u)^T (k y)
                        if constexpr (D == 2) {
                            v[0] = fma_(ua[q][0], ky[0], v[0]);
                            v[1] = fma_(ua[q][1], ky[0], fma_(ua[q][2], ky[1], v[1]));
                        } else {
                            v[0] = fma_(ua[q][0], ky[0], v[0]);
                            v[1] = fma_(ua[q][1], ky[0], fma_(ua[q][3], ky[1], v[1]));
                            v[2] = fma_(ua[q][2], ky[0], fma_(ua[q][4], ky[1], fma_(ua[q][5], ky[2], v[2])));
                        }
                    }
                }
#pragma unroll
                for (int d = 0; d < D; ++d) vs[d][u] = v[d];
            }
            if (NEED_GX) {
                static_assert(U == 4, "four points of a row are reduced together");
                // 2 coordinates of the four points in one reduction of 8 values, a third one in a reduction of 4
                T eight[8];
#pragma unroll
                for (int u = 0; u < 4; ++u) { eight[u] = vs[0][u]; eight[4 + u] = vs[1][u]; }
                const T s8 = cw_row_sums<T, 8>(eight, lane);
                {
                    const int i = cw_sum_index<8>(lane), n = n0 + (i & 3) * 4 + row;
                    if ((lane & 1) == 0 && n < n_end) atomic_add(&point_grad[(n - chunk_begin) * D + (i >> 2)], s8);
                }
                if constexpr (D == 3) {
                    const T s4 = cw_row_sums<T, 4>(vs[2], lane);
                    const int n = n0 + cw_sum_index<4>(lane) * 4 + row;
                    if ((lane & 3) == 0 && n < n_end) atomic_add(&point_grad[(n - chunk_begin) * D + 2], s4);
                }
            }
        }
    }
    if (NEED_GM) {
        // over the rows of the wavefront, then over the wavefronts that shared the slice; one atomic per scalar
#pragma unroll
        for (int q = 0; q < Q; ++q)
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                T v = rs[q][i];
                v += __shfl_xor(v, 16, 64);
                v += __shfl_xor(v, 32, 64);
                if (row == 0) shared_sums[(wave * 16 * Q + (wide ? col * Q : col) + q * apart) * NR + i] = v;
            }
        __syncthreads();
        constexpr int kSlice = 16 * Q * NR;
        const int first = group * WAVES * 16 * Q;               // the group's first Gaussian
        const int left = (M - first + 16 * Q - 1) / (16 * Q), slices_here = left < WAVES ? left : WAVES;
        for (int i = threadIdx.x; i < slices_here * kSlice; i += kThreads) {
            if (first + i / NR >= M) break;
            T v = shared_sums[i];
            for (int other = 1; other < share.reps; ++other) v += shared_sums[other * slices_here * kSlice + i];
            atomic_add(&sums[(size_t(bl) * M + first) * NR + i], v);
        }
    }
    if (NEED_GX) {
        __syncthreads();
        for (int i = threadIdx.x; i < points_per_chunk * D; i += kThreads) {
            const int n = chunk_begin + i / D;
            if (n >= N) continue;
            T* dst = grad_xes + (x_off + chunk_begin) * D + i;
            if (shared_points) atomic_add(dst, point_grad[i]); else *dst = point_grad[i];
        }
    }
}

// dL/dx alone, with lanes = Gaussians: every wavefront prepares 64 of them at once, where the kernel above prepares 16 Q in
// all four rows, and a workgroup's 256 leave fewer additions to a point.  Against that the kernel above reduces over 16
// lanes instead of 64: it is the faster one where preparation and additions are few (cw_backward).
constexpr int kCwUnroll = 8;

template <typename T, int D>
__global__ __launch_bounds__(kBlock) void componentwise_bwd_points_kernel(const T* __restrict__ grad_out, const T* __restrict__ mixture,
                                                                         const T* __restrict__ xes, T* __restrict__ grad_xes, int L,
                                                                         int M, int N, int Bx, int Lx, int m_groups, int first_mixture,
                                                                         int chunks, int points_per_chunk, bool shared_points,
                                                                         bool covariance_form) {
    constexpr int G = 1 + D + D * D;
    constexpr int kU = Rec<T, D>::kU;
    __shared__ T point_grad[kCwPointsMax * D];
    const T* exp2_tab = exp2_table<T>();
    int id = blockIdx.x;
    const int chunk = id % chunks; id /= chunks;
    const int group = id % m_groups;
    const int bl = first_mixture + id / m_groups;
    const int b = bl / L, l = bl - b * L;
    const int xb = b < Bx ? b : Bx - 1, xl = l < Lx ? l : Lx - 1;
    // (no readfirstlane here: with a provably uniform wavefront index the point coordinates arrive through scalar
    // loads, whose waits also cover the LDS traffic of the loop -- measured 15 % slower)
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const CwSlices share = cw_share(M, group, kWave, 4, wave);
    const int m = (group * 4 + share.slice) * kWave + lane;
    const bool valid = m < M;
    const size_t x_off = (size_t(xb) * Lx + xl) * N;
    const T* __restrict__ x_bl = xes + x_off * D;
    for (int i = threadIdx.x; i < points_per_chunk * D; i += kBlock) point_grad[i] = T(0);
    __syncthreads();                                        // (the table is complete as well)
    const int chunk_begin = chunk * points_per_chunk;
    if (share.slice >= 0) {
        T r[Rec<T, D>::kStride], ua[kU];            // ua = -amp * u: dL/dx takes k*y against it
        {
            const Derived<D> dv = derive<T, D>(mixture + (size_t(bl) * M + (valid ? m : 0)) * G, covariance_form);
            store_record<T, D>(r, dv, true, over_half_log2e<T>(dv.w * dv.norm), 0);
        }
#pragma unroll
        for (int i = 0; i < kU; ++i) ua[i] = -r[Rec<T, D>::kAmp] * r[i];
        const int per_rep = (points_per_chunk + share.reps - 1) / share.reps;
        const int n_begin = chunk_begin + share.rep * per_rep;
        int n_end = n_begin + per_rep < chunk_begin + points_per_chunk ? n_begin + per_rep : chunk_begin + points_per_chunk;
        n_end = n_end < N ? n_end : N;
        const T* __restrict__ go_col = grad_out + size_t(bl) * N * M + (valid ? m : 0);
        for (int n0 = n_begin; n0 < n_end; n0 += kCwUnroll) {
            T go[kCwUnroll], xs[kCwUnroll][D];
#pragma unroll
            for (int u = 0; u < kCwUnroll; ++u) {           // eight values in flight
                const int n = n0 + u < n_end ? n0 + u : n_end - 1;
                go[u] = go_col[size_t(n) * M];
#pragma unroll
                for (int d = 0; d < D; ++d) xs[u][d] = x_bl[size_t(n) * D + d];
            }
            T vs[kCwUnroll][D];                             // dL/dx terms of the eight points, this lane's Gaussian
#pragma unroll
            for (int u = 0; u < kCwUnroll; ++u) {
                T y[D], ky[D];
                const T q = quad_form<T, D, true>(r, xs[u], y);
                const T k = (valid && n0 + u < n_end) ? pair_exp2(-q, exp2_tab) * go[u] : T(0);
#pragma unroll
                for (int d = 0; d < D; ++d) ky[d] = k * y[d];
                // -(amp u)^T (k y)
                vs[u][0] = ua[0] * ky[0];
                if constexpr (D == 2) {
                    vs[u][1] = fma_(ua[1], ky[0], ua[2] * ky[1]);
                } else {
                    vs[u][1] = fma_(ua[1], ky[0], ua[3] * ky[1]);
                    vs[u][2] = fma_(ua[2], ky[0], fma_(ua[4], ky[1], ua[5] * ky[2]));
                }
            }
            // summed over the wavefront's Gaussians, four points at a time; the lane at the end of row r holds the total of
            // point {0, 2, 1, 3}[r] of the four
            const int row = lane >> 4;
            const int mine = ((row & 1) << 1) | (row >> 1);
#pragma unroll
            for (int u0 = 0; u0 < kCwUnroll; u0 += 4) {
                T total[D];
#pragma unroll
                for (int d = 0; d < D; ++d)
                    total[d] = wave_sum4_to_row_ends(vs[u0][d], vs[u0 + 1][d], vs[u0 + 2][d], vs[u0 + 3][d], lane);
                const int n = n0 + u0 + mine;
                if ((lane & 15) == 15 && n < n_end) {
#pragma unroll
                    for (int d = 0; d < D; ++d) atomic_add(&point_grad[(n - chunk_begin) * D + d], total[d]);
                }
            }
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < points_per_chunk * D; i += kBlock) {
        const int n = chunk_begin + i / D;
        if (n >= N) continue;
        T* dst = grad_xes + (x_off + chunk_begin) * D + i;
        if (shared_points) atomic_add(dst, point_grad[i]); else *dst = point_grad[i];
    }
}

// defined in gmc_dense.hip: the per-Gaussian epilogue of the summed backward pass serves this one as well
void launch_bwd_epilogue(const void* mixture, const void* sums, void* grad_mixture, size_t n_gaussians, int D, int dtype,
                         bool covariance_form, hipStream_t stream);
size_t dense_backward_workspace_bytes(const gmc_shape& s);

// Points per workgroup: about `wanted` workgroups for the launch, with chunks of the same size (a last chunk of a few
// points costs a workgroup's preparation), a multiple of 32 points within [kCwPoints, kCwPointsMax].
constexpr size_t kCwWanted = 2048;
struct CwChunks { int chunks, points; };
static CwChunks cw_chunks(size_t workgroups, int N, size_t wanted) {
    size_t chunks = (wanted + workgroups - 1) / workgroups;
    const size_t most = (size_t(N) + kCwPoints - 1) / kCwPoints, least = (size_t(N) + kCwPointsMax - 1) / kCwPointsMax;
    chunks = chunks > most ? most : chunks;
    chunks = chunks < least ? least : chunks;
    const int points = int(((size_t(N) + chunks - 1) / chunks + 31) / 32 * 32);
    return CwChunks{(N + points - 1) / points, points};
}

// (see componentwise_fwd_wide_kernel; `workgroups`: of the kernel with lanes = Gaussians)
static bool cw_wide_forward(const gmc_shape& s, size_t workgroups, bool wide) {
    if (s.dtype != GMC_F32) return false;
    return s.M <= (wide ? 64 : 32) ? s.N >= 16 : s.M > 64 && workgroups < 512 && s.N >= (wide ? 96 : 128);
}

template <typename T, int D>
static int cw_forward(const T* mixture, const T* xes, T* out, const gmc_shape& s, bool cov, hipStream_t st) {
    const size_t BL = size_t(s.B) * s.L;
    if (BL == 0 || s.N == 0 || s.M == 0) return GMC_OK;
    const int m_tiles = (s.M + kBlock - 1) / kBlock, chunks = (s.N + kCwPoints - 1) / kCwPoints;
    const size_t per_mixture = size_t(m_tiles) * chunks, at_once = max_workgroups(kBlock) / per_mixture;
    if (at_once == 0) return GMC_E_SHAPE;
    if constexpr (sizeof(T) == 4) {
        constexpr int Q = 4, kTileG = kWave * Q;
        const bool wide = s.M % Q == 0 && (uintptr_t(out) & 15) == 0;
        if (cw_wide_forward(s, BL * per_mixture, wide)) {
            const int tiles = (s.M + kTileG - 1) / kTileG;
            size_t wide_chunks = (kCwWanted + BL * tiles - 1) / (BL * tiles);
            const size_t most = s.N < 64 ? 1 : size_t(s.N) / 32;
            if (wide_chunks > most) wide_chunks = most;
            const int points = int(((s.N + wide_chunks - 1) / wide_chunks + 31) / 32 * 32);
            wide_chunks = (size_t(s.N) + points - 1) / points;
            const size_t per_wide = size_t(tiles) * wide_chunks, wide_at_once = max_workgroups(kBlock) / per_wide;
            for (size_t first = 0; first < BL; first += wide_at_once) {
                const dim3 grid(unsigned((BL - first < wide_at_once ? BL - first : wide_at_once) * per_wide));
#define GMC_CW(W) componentwise_fwd_wide_kernel<D, W><<<grid, dim3(kBlock), 0, st>>>( \
                    mixture, xes, out, s.L, s.M, s.N, s.Bx, s.Lx, tiles, int(first), int(wide_chunks), points, cov)
                if (wide) GMC_CW(true); else GMC_CW(false);
#undef GMC_CW
            }
            return hipGetLastError() == hipSuccess ? GMC_OK : GMC_E_LAUNCH;
        }
    }
    for (size_t first = 0; first < BL; first += at_once)
        componentwise_fwd_kernel<T, D><<<dim3(unsigned((BL - first < at_once ? BL - first : at_once) * per_mixture)), dim3(kBlock), 0, st>>>(
            mixture, xes, out, s.L, s.M, s.N, s.Bx, s.Lx, m_tiles, int(first), chunks, cov);
    return hipGetLastError() == hipSuccess ? GMC_OK : GMC_E_LAUNCH;
}

template <typename T, int D, int Q, int WAVES = 4>
static int cw_backward_q(const T* grad_out, const T* mixture, const T* xes, T* grad_mixture, T* grad_xes, T* sums,
                       const gmc_shape& s, bool gm, bool gx, bool wide, bool cov, hipStream_t st) {
    constexpr int G = 1 + D + D * D;
    constexpr int NR = 1 + D + D * (D + 1) / 2;
    const size_t BL = size_t(s.B) * s.L;
    const size_t n_g = BL * s.M, n_x = size_t(s.Bx) * s.Lx * s.N * D;
    if (BL == 0) return GMC_OK;
    constexpr int kGroup = WAVES * 16 * Q;
    const int m_groups = (s.M + kGroup - 1) / kGroup;
    const CwChunks c = cw_chunks(BL * (m_groups > 0 ? m_groups : 1), s.N > 0 ? s.N : 1, kCwWanted);
    const int chunks = c.chunks, points_per_chunk = c.points;
    // dL/dx of a point is stored by the one workgroup that sees all its Gaussians, and added atomically to zeros when
    // several do (more than one group of four slices, or points shared by several mixtures)
    const bool shared_points = m_groups > 1 || size_t(s.Bx) * s.Lx != BL;
    if (s.N == 0 || s.M == 0) {
        zero2_async(grad_mixture, gm ? n_g * G : 0, grad_xes, gx ? n_x : 0, st);
        return hipGetLastError() == hipSuccess ? GMC_OK : GMC_E_LAUNCH;
    }
    zero2_async(sums, gm ? n_g * NR : 0, grad_xes, gx && shared_points ? n_x : 0, st);
    // (as many mixtures a launch as its threads allow: more than one launch from 2^24 groups of Gaussians and points on)
    const size_t per_mixture = size_t(m_groups) * chunks, at_once = max_workgroups(WAVES * kWave) / per_mixture;
    if (at_once == 0) return GMC_E_SHAPE;
    for (size_t first = 0; first < BL; first += at_once) {
        const dim3 grid(unsigned((BL - first < at_once ? BL - first : at_once) * per_mixture));
#define GMC_CW(GM, GX) componentwise_bwd_kernel<T, D, Q, WAVES, GM, GX><<<grid, dim3(WAVES * kWave), 0, st>>>( \
            grad_out, mixture, xes, sums, grad_xes, s.L, s.M, s.N, s.Bx, s.Lx, m_groups, int(first), chunks, points_per_chunk, \
            shared_points, wide, cov)
        if constexpr (WAVES > 4) {
            GMC_CW(true, true);
        } else {
            if (gm && gx) GMC_CW(true, true);
            else if (gm) GMC_CW(true, false);
            else if (gx) GMC_CW(false, true);
        }
#undef GMC_CW
    }
    if (gm) launch_bwd_epilogue(mixture, sums, grad_mixture, n_g, D, s.dtype, cov, st);
    return hipGetLastError() == hipSuccess ? GMC_OK : GMC_E_LAUNCH;
}

template <typename T, int D>
static int cw_backward_points(const T* grad_out, const T* mixture, const T* xes, T* grad_xes, const gmc_shape& s, bool cov,
                              hipStream_t st) {
    const size_t BL = size_t(s.B) * s.L, n_x = size_t(s.Bx) * s.Lx * s.N * D;
    if (BL == 0 || s.N == 0) return GMC_OK;
    const int m_groups = (s.M + kBlock - 1) / kBlock;
    const CwChunks c = cw_chunks(BL * m_groups, s.N, kCwWanted);
    const bool shared_points = m_groups > 1 || size_t(s.Bx) * s.Lx != BL;
    if (shared_points) zero_async(grad_xes, n_x, st);
    const size_t per_mixture = size_t(m_groups) * c.chunks, at_once = max_workgroups(kBlock) / per_mixture;
    if (at_once == 0) return GMC_E_SHAPE;
    for (size_t first = 0; first < BL; first += at_once)
        componentwise_bwd_points_kernel<T, D><<<dim3(unsigned((BL - first < at_once ? BL - first : at_once) * per_mixture)), dim3(kBlock), 0, st>>>(
            grad_out, mixture, xes, grad_xes, s.L, s.M, s.N, s.Bx, s.Lx, m_groups, int(first), c.chunks, c.points, shared_points, cov);
    return hipGetLastError() == hipSuccess ? GMC_OK : GMC_E_LAUNCH;
}

template <typename T, int D>
static int cw_backward(const T* grad_out, const T* mixture, const T* xes, T* grad_mixture, T* grad_xes, T* sums,
                       const gmc_shape& s, bool gm, bool gx, bool cov, hipStream_t st) {
    const size_t BL = size_t(s.B) * s.L, groups = (size_t(s.M) + 63) / 64;
    const bool shared = size_t(s.Bx) * s.Lx != BL;
    // dL/dx alone: lanes = Gaussians where a Gaussian's preparation serves few points, where additions of several mixtures
    // meet on a point, or where the launch is small (more than one group: a zero fill and additions instead of stores).
    // Lanes = Gaussians / the 4 x 16 layout, us: 882 x 1179 Gaussians at 2 points, 3-D, float64 68 / 121; 2170 x 427 at 18
    // points that all share 93 / 286; 9 x 120 at 900 8.7 / 10.1; but 800 x 128 at 784 114 / 88, and with at most 64
    // Gaussians (one group) the 4 x 16 layout takes 0.65 to 1.05 of the time.
    if (!gm && gx && groups > 1 && (s.N <= 128 || shared || BL * groups * ((size_t(s.N) + 63) / 64) < 512))
        return cw_backward_points<T, D>(grad_out, mixture, xes, grad_xes, s, cov, st);
    // Both gradients, points shared by many mixtures: sixteen wavefronts a workgroup, so that 256 Gaussians make one addition
    // to a point.  Four / sixteen, us (2-D): 2170 x 427 Gaussians at 18 points 321 / 139, 728 x 153 at 17 53 / 29, float64
    // 256 x 1432 at 19 166 / 84; where fewer than 256 additions meet on a point four are as fast or faster.  (3-D in double:
    // the registers of sixteen wavefronts do not hold a Gaussian's sums.)
    if constexpr (sizeof(T) == 4 || D == 2) {
        if (gm && gx && shared && groups > 2 && BL * groups >= 256 * size_t(s.Bx) * s.Lx)
            return cw_backward_q<T, D, 1, 16>(grad_out, mixture, xes, grad_mixture, grad_xes, sums, s, gm, gx, true, cov, st);
    }
    if constexpr (sizeof(T) == 4) {
        if (cw_two_per_lane<T>(s)) {
            const bool wide = s.M % 2 == 0 && (uintptr_t(grad_out) & (2 * sizeof(T) - 1)) == 0;
            return cw_backward_q<T, D, 2>(grad_out, mixture, xes, grad_mixture, grad_xes, sums, s, gm, gx, wide, cov, st);
        }
    }
    return cw_backward_q<T, D, 1>(grad_out, mixture, xes, grad_mixture, grad_xes, sums, s, gm, gx, true, cov, st);
}

}  // namespace gmc

extern "C" {

int gmc_eval_componentwise_fwd(const void* mixture, const void* xes, void* out, const gmc_shape* shape, int covariance_form,
                               void* stream) {
    const int rc = gmc::check_shape(shape);
    if (rc != GMC_OK) return rc;
    if (size_t(shape->B) * shape->L * shape->N * shape->M == 0) return GMC_OK;
    if (!mixture || !xes || !out) return GMC_E_NULL;
    const bool cov = covariance_form != 0;
#define ARGS(T) (const T*)mixture, (const T*)xes, (T*)out, *shape, cov, (hipStream_t)stream
    if (shape->dtype == GMC_F32) return shape->D == 2 ? gmc::cw_forward<float, 2>(ARGS(float)) : gmc::cw_forward<float, 3>(ARGS(float));
    return shape->D == 2 ? gmc::cw_forward<double, 2>(ARGS(double)) : gmc::cw_forward<double, 3>(ARGS(double));
#undef ARGS
}

int gmc_eval_componentwise_bwd(const void* grad_out, const void* mixture, const void* xes, void* grad_mixture,
                               void* grad_xes, void* workspace, size_t workspace_bytes, const gmc_shape* shape,
                               int need_grad_mixture, int need_grad_xes, int covariance_form, void* stream) {
    const int rc = gmc::check_shape(shape);
    if (rc != GMC_OK) return rc;
    const bool gm = need_grad_mixture != 0, gx = need_grad_xes != 0;
    if (!gm && !gx) return GMC_OK;
    const size_t n_g = size_t(shape->B) * shape->L * shape->M;
    const size_t n_x = size_t(shape->Bx) * shape->Lx * shape->N;
    if (gm && n_g > 0 && !grad_mixture) return GMC_E_NULL;
    if (gx && n_x > 0 && !grad_xes) return GMC_E_NULL;
    if (n_g > 0 && n_x > 0 && (!grad_out || !mixture || !xes)) return GMC_E_NULL;
    if (gm && n_g > 0 && n_x > 0) {
        if (workspace_bytes < gmc::dense_backward_workspace_bytes(*shape)) return GMC_E_WORKSPACE;
        if (!workspace) return GMC_E_NULL;
    }
    const bool cov = covariance_form != 0;
#define ARGS(T) (const T*)grad_out, (const T*)mixture, (const T*)xes, (T*)grad_mixture, (T*)grad_xes, (T*)workspace, *shape, gm, gx, cov, (hipStream_t)stream
    if (shape->dtype == GMC_F32) return shape->D == 2 ? gmc::cw_backward<float, 2>(ARGS(float)) : gmc::cw_backward<float, 3>(ARGS(float));
    return shape->D == 2 ? gmc::cw_backward<double, 2>(ARGS(double)) : gmc::cw_backward<double, 3>(ARGS(double));
#undef ARGS
}

}  // extern "C"
