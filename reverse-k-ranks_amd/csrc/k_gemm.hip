// k_gemm.hip -- score kernels with the reference's sequential FP32 rule.
//
// Every score s(a, b) = sum_{k=0}^{K-1} a_k * b_k is evaluated as the
// reference's InnerProduct (src/include/alg/SpaceInnerProduct.hpp:14-20):
// one accumulator per output, k ascending, each product rounded to FP32
// and then added with FP32 rounding.  The library is compiled with
// -ffp-contract=off, so no product is fused into an FMA; the results are
// bit-identical to a scalar C loop.  That is why these are SIMT register-
// tiled kernels (v_mul_f32 + v_add_f32), not MFMA: matrix cores sum in an
// order of their own and cannot reproduce the rule.
//
// Tiling (gfx950, wave64): 256 threads as a 16 x 16 grid; each thread owns
// an 8 x 8 block of a 128 x 128 tile, split as rows {4ty..4ty+3} and
// {64+4ty..64+4ty+3} (same for columns) so that every ds_read_b128 of a
// wave covers 256 contiguous bytes.  K advances in chunks of 16 staged
// through LDS in k-major layout, double-buffered.  The bound is VALU issue,
// 128 instructions per thread and k-step: one wave issues at most one every
// 4.9 cycles, two or more ready waves one per 2.16 cycles and SIMD (a probe of
// independent v_mul / v_add).  Three waves per SIMD (156 VGPRs) cover each
// other's LDS reads and barriers; the tile's loads carry no bounds branches
// and few address registers, which a fourth wave (128 VGPRs) still spills.
// 40,000 x 50,000 x 150: 13.6 -> 11.3 ms, 26.4e12 products/s, 2.28 cycles per
// instruction at the 1.97 GHz the card holds under this load.
#include "rkr_internal.hpp"

namespace rkr {
namespace {

constexpr int BM = 128, BN = 128, KC = 16, NT = 256;
constexpr int LDS_PAD = 4;  // k-major rows of BM + pad floats

// 16-byte aligned rows, so a thread's four values are one ds_read_b128.
struct alignas(16) TileSmem {
    float a[2][KC][BM + LDS_PAD];
    float b[2][KC][BN + LDS_PAD];
};

// One thread's share of the staging of a 128-row operand: rows t / 4 and
// t / 4 + 64, the four k's at 4 (t % 4) of every chunk.  Rows past n_rows read
// the last row (their outputs are never stored or counted) and columns past
// ld the row's last four (never computed: ld >= K).
// GATHER: row r of the operand is row rows[r] of X.
template <bool GATHER>
struct ChunkLoader {
    const float *base;  // the tile's first row (X itself when gathered)
    const float *p[GATHER ? 2 : 1];
    uint32_t off[GATHER ? 1 : 2];
    int32_t ld;
    __device__ __forceinline__ ChunkLoader(const float *__restrict__ X, const int32_t *__restrict__ rows, int64_t r0,
                                           int64_t n_rows, int32_t ld_)
        : base(X + (GATHER ? 0 : r0 * ld_)), ld(ld_) {
        const int last = (int)min((int64_t)(BM - 1), n_rows - 1 - r0);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int r = min((int)(threadIdx.x >> 2) + h * 64, last);
            if constexpr (GATHER) p[h] = X + (int64_t)rows[r0 + r] * ld;
            else off[h] = (uint32_t)r * (uint32_t)ld;
        }
    }
    template <int NH>  // 64 NH rows
    __device__ __forceinline__ void load(int32_t k0, float4 (&reg)[NH]) const {
        const uint32_t k = (uint32_t)min(k0 + (int32_t)(threadIdx.x & 3) * 4, ld - 4);
#pragma unroll
        for (int h = 0; h < NH; ++h) {
            if constexpr (GATHER) reg[h] = *reinterpret_cast<const float4 *>(p[h] + k);
            else reg[h] = *reinterpret_cast<const float4 *>(base + (off[h] + k));
        }
    }
};

template <int NH>
__device__ __forceinline__ void store_chunk(float (*dst)[BM + LDS_PAD], const float4 (&reg)[NH]) {
    const int t = threadIdx.x;
    const int kq = (t & 3) * 4;
#pragma unroll
    for (int h = 0; h < NH; ++h) {
        const int m = (t >> 2) + h * 64;
        dst[kq + 0][m] = reg[h].x;
        dst[kq + 1][m] = reg[h].y;
        dst[kq + 2][m] = reg[h].z;
        dst[kq + 3][m] = reg[h].w;
    }
}

// A thread's operands of one k-step: 8 rows of A, TN (8 or 4) of B.
template <int TN>
struct StepFrag {
    float4 a0, a1, b[TN / 4];
    __device__ __forceinline__ void read(const float *__restrict__ pa, const float *__restrict__ pb) {
        a0 = *reinterpret_cast<const float4 *>(pa);
        a1 = *reinterpret_cast<const float4 *>(pa + 64);
#pragma unroll
        for (int h = 0; h < TN / 4; ++h) b[h] = *reinterpret_cast<const float4 *>(pb + 64 * h);
    }
    __device__ __forceinline__ void add_to(float (&acc)[8][TN]) const {
        const float av[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
        float bv[TN];
#pragma unroll
        for (int h = 0; h < TN / 4; ++h) {
            bv[4 * h] = b[h].x;
            bv[4 * h + 1] = b[h].y;
            bv[4 * h + 2] = b[h].z;
            bv[4 * h + 3] = b[h].w;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const float p = av[i] * bv[j];
                acc[i][j] = acc[i][j] + p;
            }
    }
};

// acc[i][j] = score(A row i of the tile, B row j of the tile) over k < K; with
// TN = 4 the tile has the first 64 of its B rows only.
template <bool GATHER, int TN = 8>
__device__ __forceinline__ void tile_scores(TileSmem &sm, const float *__restrict__ A,
                                            const int32_t *__restrict__ a_rows, int64_t m0, int64_t M,
                                            int32_t lda, const float *__restrict__ B, int64_t n0, int64_t N,
                                            int32_t ldb, int32_t K, float (&acc)[8][TN]) {
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = 0.0f;

    const ChunkLoader<GATHER> la(A, a_rows, m0, M, lda);
    const ChunkLoader<false> lb(B, nullptr, n0, N, ldb);
    float4 ra[2], rb[TN / 4];
    const int nchunk = (K + KC - 1) / KC;
    la.load(0, ra);
    lb.load(0, rb);
    store_chunk(sm.a[0], ra);
    store_chunk(sm.b[0], rb);
    __syncthreads();
    for (int c = 0; c < nchunk; ++c) {
        const int buf = c & 1;
        const int k0 = c * KC;
        // the next chunk's loads are in flight while this one is computed (the
        // last chunk's are its own again, unused)
        la.load(min(k0 + KC, (nchunk - 1) * KC), ra);
        lb.load(min(k0 + KC, (nchunk - 1) * KC), rb);
        const float *pa = &sm.a[buf][0][ty * 4], *pb = &sm.b[buf][0][tx * 4];
        constexpr int ROW = BM + LDS_PAD;
        static_assert(BM == BN, "one row stride for both operands");
        const int kend = min(KC, K - k0);
#pragma unroll 4
        for (int kk = 0; kk < kend; ++kk) {
            StepFrag<TN> f;
            f.read(pa, pb);
            f.add_to(acc);
            pa += ROW;
            pb += ROW;
        }
        if (c + 1 < nchunk) {
            store_chunk(sm.a[buf ^ 1], ra);
            store_chunk(sm.b[buf ^ 1], rb);
        }
        __syncthreads();
    }
}

__device__ __forceinline__ int tile_row(int i) { return (i < 4) ? ((threadIdx.x >> 4) * 4 + i) : (64 + (threadIdx.x >> 4) * 4 + i - 4); }
__device__ __forceinline__ int tile_col(int j) { return (j < 4) ? ((threadIdx.x & 15) * 4 + j) : (64 + (threadIdx.x & 15) * 4 + j - 4); }

// Workgroups go to the 8 XCDs in turn, each with its own L2: block p takes
// logical tile (p % 8) * per + p / 8, so an XCD runs one contiguous eighth of
// the tiles, and logical tiles walk the columns of a band of kBand tile rows,
// the band's rows first, so the tiles an XCD runs at one time share their A
// rows and a few B column blocks.
constexpr int64_t kBand = 8;

__device__ __forceinline__ bool tile_of_block(int64_t n_tiles_m, int64_t n_tiles_n, int64_t &tm, int64_t &tn) {
    const int64_t n_tiles = n_tiles_m * n_tiles_n, per = (n_tiles + 7) / 8;
    const int64_t t = (int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (t >= n_tiles || (int64_t)(blockIdx.x >> 3) >= per) return false;
    const int64_t band = t / (kBand * n_tiles_n), in = t - band * (kBand * n_tiles_n);
    const int64_t rows = min(kBand, n_tiles_m - band * kBand);
    tm = band * kBand + in % rows;
    tn = in / rows;
    return true;
}

// ROW_M: C[m * ldc + n], else C[n * ldc + m].  vec: rows of C start 16-byte
// aligned, so four neighbouring outputs are one store.
template <bool ROW_M, int TN>
__device__ __forceinline__ void store_tile(TileSmem &sm, const float *__restrict__ A, int64_t M, int32_t lda,
                                           const float *__restrict__ B, int64_t N, int32_t ldb, int32_t K,
                                           float *__restrict__ C, int64_t ldc, int vec, int64_t m0, int64_t n0) {
    float acc[8][TN];
    tile_scores<false, TN>(sm, A, nullptr, m0, M, lda, B, n0, N, ldb, K, acc);
    // outer index o runs over C's rows, inner over the contiguous direction
    constexpr int NO = ROW_M ? 8 : TN, NI = ROW_M ? TN : 8;
    const int64_t o0 = ROW_M ? m0 : n0, i0 = ROW_M ? n0 : m0, n_o = ROW_M ? M : N, n_i = ROW_M ? N : M;
#pragma unroll
    for (int o = 0; o < NO; ++o) {
        const int64_t r = o0 + (ROW_M ? tile_row(o) : tile_col(o));
        if (r >= n_o) continue;
#pragma unroll
        for (int h = 0; h < NI / 4; ++h) {
            const int64_t q = i0 + (ROW_M ? tile_col(4 * h) : tile_row(4 * h));
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if constexpr (ROW_M) v[j] = acc[o][4 * h + j];
                else v[j] = acc[4 * h + j][o];
            }
            float *dst = C + r * ldc + q;
            if (vec && q + 3 < n_i) {
                *reinterpret_cast<float4 *>(dst) = make_float4(v[0], v[1], v[2], v[3]);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (q + j < n_i) dst[j] = v[j];
            }
        }
    }
}

// A last column block of up to 64 columns takes half the products of a whole
// one: batches of 17 to 64 queries, and the 44 columns that 300 queries leave.
// 100,003 users x 145 dims: 300 queries 269 -> 249 us, 48 queries 115 -> 68.
template <bool ROW_M>
__global__ void __launch_bounds__(NT, 3) k_scores_store(const float *__restrict__ A, int64_t M, int32_t lda,
                                                     const float *__restrict__ B, int64_t N,
                                                     int32_t ldb, int32_t K, float *__restrict__ C, int64_t ldc,
                                                     int vec, int64_t n_tiles_m, int64_t n_tiles_n, uint64_t *t) {
    stamp(t);
    __shared__ TileSmem sm;
    int64_t tm, tn;
    if (!tile_of_block(n_tiles_m, n_tiles_n, tm, tn)) return;
    const int64_t m0 = tm * BM, n0 = tn * BN;
    if (N - n0 <= BN / 2) store_tile<ROW_M, 4>(sm, A, M, lda, B, N, ldb, K, C, ldc, vec, m0, n0);
    else store_tile<ROW_M, 8>(sm, A, M, lda, B, N, ldb, K, C, ldc, vec, m0, n0);
}

// Persistent refinement count.  Work unit = (block of 128 refine rows,
// group of item tiles).  Each unit adds, for every row r of its
// block, #{items p in the group : score(user(r), p) > thr(r)} to cnt[r].
// A group is as many tiles (up to kGroup) as leave every workgroup of the grid
// a unit: with table columns at every top rank there are often fewer than 128
// rows in all, and groups of 8 tiles then used 98 of 256 CUs (92 rows against
// 100k items, 150 dims: 300 us; one tile a unit: 94 us).
//
// OCC workgroups per CU: 3 hide the start of a unit, its gather of rows, when
// units are single tiles (300 rows x 100k items x 128 dims: 0.18 ms, with 2
// 0.245); over many rows 2 are faster, the three run in step and the card
// clocks lower (125k rows x 21k items x 157 dims: 13.2 ms, with 3 15.7).
constexpr int kGroup = 8;  // a thread counts at most 8 per tile and row: 8 * kGroup < 256

template <int OCC>
__global__ void __launch_bounds__(NT, OCC) k_refine_count(const float *__restrict__ users, const float *__restrict__ items,
                                                     int64_t n_item, int32_t ld, int32_t K,
                                                     const int32_t *__restrict__ rows_user,
                                                     const float *__restrict__ rows_thr,
                                                     const int32_t *__restrict__ n_rows_dev, int64_t max_rows,
                                                     int32_t *__restrict__ cnt, uint64_t *t) {
    stamp(t);
    __shared__ TileSmem sm;
    __shared__ int32_t red[BM];
    __shared__ float s_thr[BM];
    const int64_t n_rows = min((int64_t)*n_rows_dev, max_rows);
    const int64_t n_rb = (n_rows + BM - 1) / BM;
    const int64_t n_it = (n_item + BN - 1) / BN;
    const int64_t grp = max((int64_t)1, min((int64_t)kGroup, n_rb * n_it / gridDim.x));
    const int64_t n_grp = (n_it + grp - 1) / grp;
    const int64_t n_units = n_rb * n_grp;
    for (int64_t unit = blockIdx.x; unit < n_units; unit += gridDim.x) {
        const int64_t rb = unit / n_grp, g = unit % n_grp;
        const int64_t m0 = rb * BM;
        if (threadIdx.x < BM) {
            const int64_t m = m0 + threadIdx.x;
            s_thr[threadIdx.x] = m < n_rows ? rows_thr[m] : 0.0f;  // read after tile_scores' barriers
            red[threadIdx.x] = 0;
        }
        // the thread's eight row counts, a byte each (at most 8 per tile, 64
        // per unit): registers are short beside the tile
        uint32_t c[2] = {0u, 0u};
        const int64_t t_end = min((g + 1) * grp, n_it);
        for (int64_t it = g * grp; it < t_end; ++it) {
            const int64_t n0 = it * BN;
            float acc[8][8];
            tile_scores<true>(sm, users, rows_user, m0, n_rows, ld, items, n0, n_item, ld, K, acc);
            const int n_in = (int)min((int64_t)BN, n_item - n0);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float thr = s_thr[tile_row(i)];
                uint32_t v = 0;
#pragma unroll
                for (int j = 0; j < 8; ++j) v += (tile_col(j) < n_in && acc[i][j] > thr) ? 1u : 0u;
                c[i >> 2] += v << (8 * (i & 3));
            }
        }
        // reduce over the 16 threads that share each row
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int32_t v = (int32_t)((c[i >> 2] >> (8 * (i & 3))) & 0xFFu);
            if (v) atomicAdd(&red[tile_row(i)], v);
        }
        __syncthreads();
        if (threadIdx.x < BM) {
            const int64_t m = m0 + threadIdx.x;
            if (m < n_rows && red[threadIdx.x]) atomicAdd(&cnt[m], red[threadIdx.x]);
        }
        __syncthreads();
    }
}

// Small-batch <u, q>: one wave per 64-user panel, lane = user.  Users are
// stored as panels [p][k][lane] so every k step is one coalesced 256-byte
// load, 16 of them in flight ahead of the sums; query values are uniform and
// come through the scalar cache.  With bk also #{T > score} of every pair, the
// NQ searches of a user side by side so their loads overlap.
// Bound: the panels' bytes (7 queries x 250k users x 128 dims, 128 MB: 74 us
// with one load in flight and the queries in LDS, now 33; 16 x 100k x 150, 60 MB: 133 us, now 44).
constexpr int GC = 16;

template <int NQ>
__global__ void __launch_bounds__(NT) k_gemv_panels(const float *__restrict__ usersT, int64_t n_user, int32_t ld,
                                                    int32_t K, const float *__restrict__ q, int32_t nq,
                                                    float *__restrict__ qip, const float *__restrict__ table, int32_t S,
                                                    uint32_t *__restrict__ bk, uint64_t *t) {
    stamp(t);
    const int lane = threadIdx.x & 63;
    const int64_t panel = (int64_t)blockIdx.x * (NT / 64) + (threadIdx.x >> 6);
    const int64_t u = panel * 64 + lane;
    if (panel * 64 >= n_user) return;
    const float *src = usersT + panel * (int64_t)ld * 64 + lane;
    float acc[NQ];
#pragma unroll
    for (int b = 0; b < NQ; ++b) acc[b] = 0.0f;
    float x[GC], y[GC];
    auto load = [&](int32_t k0, float (&v)[GC]) {
#pragma unroll
        for (int j = 0; j < GC; ++j) v[j] = src[(int64_t)min(k0 + j, K - 1) * 64];
    };
    load(0, x);
    int32_t k0 = 0;
    for (; k0 + GC <= K; k0 += GC) {
        load(k0 + GC, y);  // past the last term: its value again, unused
#pragma unroll
        for (int b = 0; b < NQ; ++b) {
            const float *qb = q + min(b, nq - 1) * (int64_t)ld + k0;
#pragma unroll
            for (int j = 0; j < GC; ++j) {
                const float p = x[j] * qb[j];
                acc[b] = acc[b] + p;
            }
        }
#pragma unroll
        for (int j = 0; j < GC; ++j) x[j] = y[j];
    }
#pragma unroll
    for (int j = 0; j < GC; ++j)
        if (k0 + j < K)
#pragma unroll
            for (int b = 0; b < NQ; ++b) {
                const float p = x[j] * q[min(b, nq - 1) * (int64_t)ld + k0 + j];
                acc[b] = acc[b] + p;
            }
    if (u >= n_user) return;
#pragma unroll
    for (int b = 0; b < NQ; ++b)
        if (b < nq) qip[(int64_t)b * n_user + u] = acc[b];
    if (!bk) return;
    const float *row = table + u * (int64_t)S;
    int32_t pos[NQ];
#pragma unroll
    for (int b = 0; b < NQ; ++b) pos[b] = 0;
    for (int32_t step = 1 << (31 - __clz(S)); step > 0; step >>= 1)
#pragma unroll
        for (int b = 0; b < NQ; ++b) {
            const int32_t at = pos[b] + step;
            const float v = row[min(at, S) - 1];
            pos[b] = at <= S && v > acc[b] ? at : pos[b];
        }
#pragma unroll
    for (int b = 0; b < NQ; ++b)
        if (b < nq) bk[(int64_t)b * n_user + u] = (uint32_t)pos[b] | (uint32_t)pos[b] << 16;
}

__global__ void k_make_panels(const float *__restrict__ users, int64_t n_user, int32_t ld, float *__restrict__ usersT) {
    const int64_t n_panel = (n_user + 63) / 64;
    const int64_t total = n_panel * ld * 64;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t lane = i & 63;
        const int64_t k = (i >> 6) % ld;
        const int64_t p = (i >> 6) / ld;
        const int64_t u = p * 64 + lane;
        usersT[i] = u < n_user ? users[u * ld + k] : 0.0f;
    }
}

}  // namespace

hipError_t launch_scores_store(hipStream_t s, const float *A, int64_t M, int32_t lda,
                               const float *B, int64_t N, int32_t ldb, int32_t K, float *C, int64_t ldc,
                               bool c_row_major_m, uint64_t *t) {
    if (M <= 0 || N <= 0) return hipSuccess;
    const int64_t tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN;
    const dim3 grid((unsigned)((tm * tn + 7) / 8 * 8));
    const int vec = ldc % 4 == 0 && reinterpret_cast<uintptr_t>(C) % 16 == 0 ? 1 : 0;
    if (c_row_major_m)
        hipLaunchKernelGGL(k_scores_store<true>, grid, dim3(NT), 0, s, A, M, lda, B, N, ldb, K, C, ldc, vec, tm, tn, t);
    else
        hipLaunchKernelGGL(k_scores_store<false>, grid, dim3(NT), 0, s, A, M, lda, B, N, ldb, K, C, ldc, vec, tm, tn, t);
    return hipGetLastError();
}

hipError_t launch_refine_count(hipStream_t s, const float *users, const float *items, int64_t n_item, int32_t ld,
                               int32_t K, const int32_t *rows_user, const float *rows_thr, const int32_t *n_rows_dev,
                               int64_t max_rows, int32_t *cnt, bool many, uint64_t *t) {
    if (max_rows <= 0 || n_item <= 0) return hipSuccess;
    int dev = 0, n_cu = 256;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev);
    const int64_t n_it = (n_item + BN - 1) / BN;
    const int64_t max_units = ((max_rows + BM - 1) / BM) * n_it;
    many = many && max_units >= (int64_t)kGroup * n_cu * 2;
    const dim3 grid((unsigned)std::min<int64_t>(max_units, (int64_t)n_cu * (many ? 2 : 3)));
    if (many)
        hipLaunchKernelGGL(k_refine_count<2>, grid, dim3(NT), 0, s, users, items, n_item, ld, K, rows_user, rows_thr,
                           n_rows_dev, max_rows, cnt, t);
    else
        hipLaunchKernelGGL(k_refine_count<3>, grid, dim3(NT), 0, s, users, items, n_item, ld, K, rows_user, rows_thr,
                           n_rows_dev, max_rows, cnt, t);
    return hipGetLastError();
}

hipError_t launch_gemv_panels(hipStream_t s, const float *usersT, int64_t n_user, int32_t ld, int32_t K,
                              const float *q, int32_t nq, float *qip, const float *table, int32_t S, uint32_t *bk,
                              uint64_t *t) {
    if (n_user <= 0 || nq <= 0) return hipSuccess;
    if (nq > 16 || (bk && (!table || S <= 0))) return hipErrorInvalidValue;
    const int64_t n_panel = (n_user + 63) / 64;
    const dim3 grid((unsigned)((n_panel + 3) / 4)), block(NT);
#define RKR_GEMV(n) hipLaunchKernelGGL(k_gemv_panels<n>, grid, block, 0, s, usersT, n_user, ld, K, q, nq, qip, table, S, bk, t)
    if (nq <= 1) RKR_GEMV(1);
    else if (nq <= 2) RKR_GEMV(2);
    else if (nq <= 4) RKR_GEMV(4);
    else if (nq <= 8) RKR_GEMV(8);
    else RKR_GEMV(16);
#undef RKR_GEMV
    return hipGetLastError();
}

hipError_t launch_make_panels(hipStream_t s, const float *users, int64_t n_user, int32_t ld, float *usersT) {
    if (n_user <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_make_panels, dim3(2048), dim3(256), 0, s, users, n_user, ld, usersT);
    return hipGetLastError();
}

}  // namespace rkr
