// k_train.hip -- the device half of QS sample-rank training.
//
// 1. Query-rank distribution (ComputeQueryRankByComputation,
//    src/app/build-index/QueryRankByComputation.hpp:122-242, with the rank of
//    QueryRankGPU::ComputeRankOfQuery, src/app/build-index/QueryRankGPU.hpp:63-92,225-240):
//    for every user u and sample item s, rank(u, s) = #{items whose score
//    beats <u, s>} -- the lower_bound with greater<float> in u's descending
//    row.  k_rank_hist_lds (row staged in LDS) or k_rank_hist counts
//    hist[s][rank] over the users of a batch.
// 2. The sample-rank DP of FindOptimalSampleFast
//    (src/include/alg/RankBoundRefinement/FindSampleRank/OptimalSampleRankFast.hpp:160-205):
//    k_transit fills the transit-cost triangle of QueryDistribution
//    (OptimalSampleRank.hpp:233-318) from per-rank prefix sums over the
//    queries, in O(1) per pair; k_dp_layers runs the DP, k_dp_layer one layer
//    of it for more ranks than that holds in registers.
#include "rkr_internal.hpp"

#include <climits>

namespace rkr {
namespace {

// One workgroup per user row; threads take the samples.
__global__ void __launch_bounds__(256) k_rank_hist(const float *__restrict__ sorted, int64_t ld, int32_t n_item,
                                                   const float *__restrict__ q, int64_t ldq, int32_t ns,
                                                   int32_t *__restrict__ hist) {
    const int64_t u = blockIdx.x;
    const float *row = sorted + u * ld;
    for (int s = threadIdx.x; s < ns; s += blockDim.x) {
        const float x = q[u * ldq + s];
        int lo = 0, hi = n_item;  // first position whose value is not > x
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (row[mid] > x) lo = mid + 1;
            else hi = mid;
        }
        atomicAdd(hist + (int64_t)s * (n_item + 1) + lo, 1);
    }
}

// The same count with the row staged in LDS first (n_item floats of dynamic
// LDS): each binary search then reads LDS instead of issuing its ~15 dependent
// requests to the caches.  Used when the row fits the workgroup's LDS.
// With ranks the rank goes there (ranks[u * ldr + s]) and k_rank_count counts.
__global__ void __launch_bounds__(512) k_rank_hist_lds(const float *__restrict__ sorted, int64_t ld, int32_t n_item,
                                                       const float *__restrict__ q, int64_t ldq, int32_t ns,
                                                       int32_t *__restrict__ hist, uint16_t *__restrict__ ranks,
                                                       int64_t ldr) {
    extern __shared__ float srow[];
    const int64_t u = blockIdx.x;
    const float *row = sorted + u * ld;
    for (int i = threadIdx.x; i < n_item; i += blockDim.x) srow[i] = row[i];
    __syncthreads();
    for (int s = threadIdx.x; s < ns; s += blockDim.x) {
        const float x = q[u * ldq + s];
        int lo = 0, hi = n_item;  // first position whose value is not > x
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (srow[mid] > x) lo = mid + 1;
            else hi = mid;
        }
        if (ranks) ranks[u * ldr + s] = (uint16_t)lo;
        else atomicAdd(hist + (int64_t)s * (n_item + 1) + lo, 1);
    }
}

// hist[s][r] += #{u < nb : ranks[u * ldr + s] == r} for SPW samples per
// workgroup, counted in LDS (a global add per rank, 50M of them over 40 MB of
// counts at 50k users and 1000 samples, took 1.4 of 2.0 ms).
template <int SPW>
__global__ void __launch_bounds__(1024) k_rank_count(const uint16_t *__restrict__ ranks, int64_t ldr, int64_t nb,
                                                     int32_t n_item, int32_t ns, int32_t *__restrict__ hist) {
    extern __shared__ int32_t h[];  // SPW x (n_item + 1)
    const int64_t W = (int64_t)n_item + 1;
    const int32_t s0 = (int32_t)blockIdx.x * SPW;
    for (int64_t i = threadIdx.x; i < SPW * W; i += 1024) h[i] = 0;
    __syncthreads();
    for (int64_t u0 = threadIdx.x; u0 < nb; u0 += 4 * 1024) {
        uint16_t r[4][SPW];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint16_t *p = ranks + min(u0 + k * 1024, nb - 1) * ldr + s0;
            if constexpr (SPW == 4) {
                const uint2 v = *reinterpret_cast<const uint2 *>(p);
                r[k][0] = (uint16_t)v.x; r[k][1] = (uint16_t)(v.x >> 16);
                r[k][2] = (uint16_t)v.y; r[k][3] = (uint16_t)(v.y >> 16);
            } else {
                r[k][0] = *p;
            }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (u0 + k * 1024 < nb)
#pragma unroll
                for (int j = 0; j < SPW; ++j)
                    if (s0 + j < ns) atomicAdd(&h[j * W + r[k][j]], 1);
    }
    __syncthreads();
    const int32_t n = min(SPW, ns - s0);
    for (int64_t i = threadIdx.x; i < n * W; i += 1024)
        if (h[i]) hist[s0 * W + i] += h[i];
}

__device__ inline int64_t tri_off(int64_t lb) { return lb * (lb - 1) / 2; }

// T[tri_off(lb) + ub] = -End(ub) + Between(ub, lb) + End(lb) for ub < lb, where
// Between(ub, lb) = sum over queries q in [pos[ub], pos[lb]) of
// accu[q][rank_lb] - accu[q][rank_ub], read as differences of the prefix sums
// S_j(x) = sum_{q' < x} accu[q'][rank_j], which C keeps at the breakpoints:
// C[col[j'] * R + j] = S_j(pos[j']).  For one lb the threads read C's rows
// col[lb] and col[ub] at consecutive ub.
__global__ void __launch_bounds__(256) k_transit(const int64_t *__restrict__ C, int32_t Q,
                                                 const int32_t *__restrict__ pos, const int32_t *__restrict__ col,
                                                 const int64_t *__restrict__ end_cost, int32_t R,
                                                 int64_t *__restrict__ T) {
    const int64_t lb = blockIdx.x;
    if (lb < 1 || lb >= R) return;
    const int32_t pe = pos[lb];
    const int64_t *Ce = C + (int64_t)col[lb] * R;
    const int64_t el = end_cost[lb];
    int64_t *Tl = T + tri_off(lb);
    for (int64_t ub = threadIdx.x; ub < lb; ub += blockDim.x) {
        const int32_t pb = pos[ub];
        int64_t between = 0;
        if (pb < Q && pb < pe) {
            const int64_t *Cb = C + (int64_t)col[ub] * R;
            between = (Ce[lb] - Cb[lb]) - (Ce[ub] - Cb[ub]);
        }
        Tl[ub] = -end_cost[ub] + between + el;
    }
}

// One wavefront per rank r: the carried value dp_prev[r] wins ties, then the
// smallest p, as the reference's sequential loop with a strict comparison does.
__global__ void __launch_bounds__(256) k_dp_layer(const int64_t *__restrict__ T, const int64_t *__restrict__ dp_prev,
                                                  const int32_t *__restrict__ pos_prev, int32_t R,
                                                  int64_t *__restrict__ dp_cur, int32_t *__restrict__ pos_cur) {
    const int64_t r = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / 64;
    const int lane = threadIdx.x & 63;
    if (r >= R) return;  // whole wavefronts leave together
    const int64_t *Tr = T + tri_off(r);
    long long best = LLONG_MAX;
    int bp = INT_MAX;
    for (int p = lane; p < r; p += 64) {
        const long long c = dp_prev[p] + Tr[p];
        if (c < best) {
            best = c;
            bp = p;
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        const long long oc = __shfl_xor(best, off, 64);
        const int op = __shfl_xor(bp, off, 64);
        if (oc < best || (oc == best && op < bp)) {
            best = oc;
            bp = op;
        }
    }
    if (lane == 0) {
        if (bp != INT_MAX && best < dp_prev[r]) {
            dp_cur[r] = best;
            pos_cur[r] = bp;
        } else {
            dp_cur[r] = dp_prev[r];
            pos_cur[r] = pos_prev[r];
        }
    }
}

// All layers of the DP in one launch, for up to 64 MAXC ranks: one wavefront per
// rank, its row of transit costs in registers for every layer.  A layer's value
// of rank r needs the previous layer's of the ranks below r only, so there is no
// barrier between workgroups: a value is published in its layer's row, which
// starts out as kDpUnset, and a workgroup reads the rows of the workgroups before
// it until no value is unset.  Workgroups start in order, so those it waits for
// are running or done and never wait for it; the wait is bounded all the same
// (spin_max), and *err then sends the call to a launch per layer.
// Bound: per layer one trip of a value between XCDs and a wavefront's reduction.
// 511 layers of about 1100 ranks: 3.8 ms in 511 launches and 1.7 between them,
// now 1.46 in one.
template <int MAXC>
__global__ void __launch_bounds__(256) k_dp_layers(const int64_t *__restrict__ T, int32_t R, int32_t n_layer,
                                                   int64_t *dp, int32_t *__restrict__ path, int32_t spin_max,
                                                   int32_t *err) {
    constexpr int W = 4, PER = 64 * MAXC / 256;
    __shared__ long long v[2][64 * MAXC];
    __shared__ int32_t s_bad;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int32_t r0 = (int32_t)blockIdx.x * W, r = r0 + w;
    const bool live = r < R;
    long long t[MAXC];
#pragma unroll
    for (int i = 0; i < MAXC; ++i) {
        const int p = lane + 64 * i;
        t[i] = live && p < r ? T[tri_off(r) + p] : 0;
    }
    long long own = live ? dp[r] : 0;
    int32_t pos = live ? path[r] : 0;
    if (threadIdx.x == 0) s_bad = 0;
    __syncthreads();
    for (int32_t l = 1; l < n_layer; ++l) {
        long long *buf = v[l & 1];
        const int64_t *prev = dp + (int64_t)(l - 1) * R;
        long long x[PER];
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int p = (int)threadIdx.x + 256 * j;
            x[j] = p < r0 ? (long long)__hip_atomic_load(prev + p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
        }
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int p = (int)threadIdx.x + 256 * j;
            if (p >= r0) continue;
            for (int32_t n = 0; x[j] == kDpUnset && n < spin_max; ++n) {
                __builtin_amdgcn_s_sleep(1);
                x[j] = (long long)__hip_atomic_load(prev + p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            if (x[j] == kDpUnset) s_bad = 1;
            buf[p] = x[j];
        }
        if (lane == 0 && live) buf[r] = own;
        __syncthreads();
        if (s_bad) {
            if (threadIdx.x == 0) *err = 1;
            return;
        }
        long long best = LLONG_MAX;
        int bp = INT_MAX;
#pragma unroll
        for (int i = 0; i < MAXC; ++i) {
            const int p = lane + 64 * i;
            if (p < r) {
                const long long c = buf[p] + t[i];
                if (c < best) {
                    best = c;
                    bp = p;
                }
            }
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const long long oc = __shfl_xor(best, off, 64);
            const int op = __shfl_xor(bp, off, 64);
            if (oc < best || (oc == best && op < bp)) {
                best = oc;
                bp = op;
            }
        }
        if (bp != INT_MAX && best < own) {
            own = best;
            pos = bp;
        }
        if (lane == 0 && live) {
            __hip_atomic_store(dp + (int64_t)l * R + r, (int64_t)own, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            path[(int64_t)l * R + r] = pos;
        }
    }
}

}  // namespace

hipError_t launch_rank_hist(hipStream_t s, const float *sorted, int64_t ld, int64_t nb, int64_t n_item, const float *q,
                            int64_t ldq, int32_t ns, int32_t *hist, uint16_t *ranks) {
    if (nb <= 0 || ns <= 0) return hipSuccess;
    if (n_item <= 0 || n_item >= INT_MAX || nb > INT_MAX) return hipErrorInvalidValue;
    int dev = 0, lds_max = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
    if (e != hipSuccess) return e;
    const size_t lds = sizeof(float) * (size_t)n_item;
    bool use_lds = lds <= (size_t)lds_max;
    if (use_lds && hipFuncSetAttribute((const void *)k_rank_hist_lds, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)lds) != hipSuccess) {
        (void)hipGetLastError();  // a refused attribute: the row stays in global memory
        use_lds = false;
    }
    // ranks of 16 bits, and one sample's counts beside nothing else in LDS
    const size_t row_cnt = sizeof(int32_t) * ((size_t)n_item + 1);
    const bool count = use_lds && ranks && n_item < 65536 && row_cnt <= (size_t)lds_max;
    const bool four = count && 4 * row_cnt <= (size_t)lds_max;
    const void *kc = four ? (const void *)k_rank_count<4> : (const void *)k_rank_count<1>;
    const size_t lds_c = (four ? 4 : 1) * row_cnt;
    if (count && hipFuncSetAttribute(kc, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_c) != hipSuccess) {
        (void)hipGetLastError();
        ranks = nullptr;
    } else if (!count) {
        ranks = nullptr;
    }
    const int64_t ldr = rank_row(ns);
    if (use_lds)
        hipLaunchKernelGGL(k_rank_hist_lds, dim3((unsigned)nb), dim3(512), lds, s, sorted, ld, (int32_t)n_item, q, ldq,
                           ns, hist, ranks, ldr);
    else
        hipLaunchKernelGGL(k_rank_hist, dim3((unsigned)nb), dim3(256), 0, s, sorted, ld, (int32_t)n_item, q, ldq, ns,
                           hist);
    if (ranks && four)
        hipLaunchKernelGGL(k_rank_count<4>, dim3((unsigned)((ns + 3) / 4)), dim3(1024), lds_c, s, ranks, ldr, nb,
                           (int32_t)n_item, ns, hist);
    else if (ranks)
        hipLaunchKernelGGL(k_rank_count<1>, dim3((unsigned)ns), dim3(1024), lds_c, s, ranks, ldr, nb, (int32_t)n_item, ns,
                           hist);
    return hipGetLastError();
}

hipError_t launch_transit(hipStream_t s, const int64_t *C, int32_t Q, const int32_t *pos, const int32_t *col,
                          const int64_t *end_cost, int32_t R, int64_t *T) {
    if (R < 2) return hipSuccess;
    hipLaunchKernelGGL(k_transit, dim3((unsigned)R), dim3(256), 0, s, C, Q, pos, col, end_cost, R, T);
    return hipGetLastError();
}

bool dp_in_one_launch(int64_t R) { return R <= 2048; }

hipError_t launch_dp_layers(hipStream_t s, const int64_t *T, int32_t R, int32_t n_layer, int64_t *dp, int32_t *path,
                            int32_t spin_max, int32_t *err) {
    if (R <= 0 || n_layer <= 1) return hipSuccess;
    if (!dp_in_one_launch(R)) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((R + 3) / 4)), block(256);
    if (R <= 512) hipLaunchKernelGGL(k_dp_layers<8>, grid, block, 0, s, T, R, n_layer, dp, path, spin_max, err);
    else if (R <= 1024) hipLaunchKernelGGL(k_dp_layers<16>, grid, block, 0, s, T, R, n_layer, dp, path, spin_max, err);
    else hipLaunchKernelGGL(k_dp_layers<32>, grid, block, 0, s, T, R, n_layer, dp, path, spin_max, err);
    return hipGetLastError();
}

hipError_t launch_dp_layer(hipStream_t s, const int64_t *T, const int64_t *dp_prev, const int32_t *pos_prev, int32_t R,
                           int64_t *dp_cur, int32_t *pos_cur) {
    if (R <= 0) return hipSuccess;
    const int64_t waves = R;
    hipLaunchKernelGGL(k_dp_layer, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, s, T, dp_prev, pos_prev, R, dp_cur,
                       pos_cur);
    return hipGetLastError();
}

}  // namespace rkr
