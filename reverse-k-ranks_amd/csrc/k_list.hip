// k_list.hip -- the bound stage of exact output: which users a query has to
// look at, their exact scores, table buckets and the k-th bound.
//
// Every user keeps the values of up to 63 fine columns of its searched table
// row (the guard row, G_0 >= G_1 >= ... at columns col_0 < col_1 < ...).  A
// query is given one of them as its threshold t, and the users with
//     s + e >= G_t      (s their score or its estimate, e its error bound)
// are listed.  A user left out has G_t above its score, so its bucket
// b_hi = #{T > score} is past col_t.  Only the listed users get an exact score
// and a table search; when at least k of them have b_lo <= col_t, the k-th
// smallest bound beta of all users is among theirs, beta <= col_t, and every
// candidate (b_hi <= beta) is listed: beta, the candidates and the ranks are
// those of a search over every user.  A query for which that fails is answered
// by the full search instead, so t only decides how long the list is.
//
// t comes from a sample of the users, one of every stride (all of them for few
// users, where the k-th bound is then exact): the smallest column that as many
// sampled users reach for certain (s - e) as k users would need, plus a margin
// of three standard deviations, since a threshold that is too tight costs a
// full search and one that is too loose a longer list.
//
// Scores come either from the matrix cores (screened form: one BF16 product,
// |s^ - s| <= e = ||u|| cs(q) + floor, see k_screen.hip) or from the exact
// scores of the batch (plain form, e = eps of an installed table).  Where the
// items' scores lie closer together than the one product's error tells apart
// (items that share a large common part), a query is attempted again with three
// products of the high and low halves, an error 33 times smaller, and then with
// exact scores.  1M users x 1000 queries, items = mean + noise of 5%, 3% and 1% of
// it: 29, 47 and 50 ms with one product for all, now 2.3 each.
#include "rkr_internal.hpp"

namespace rkr {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int NT = 256;
constexpr int QST = 64;       // queries per LDS stage
constexpr int KPAD_LDS = 8;   // bf16 pad per LDS row
constexpr int GW = kGuardRow; // floats per guard row
static_assert(kMaxFine < GW, "a position past every fine column is a bin of its own");

union Frag {
    bf16x8 v;
    u32x4 q;
};

// #{f < 63 : row[f] > x} of a guard row (non-increasing, -inf past the fine
// columns): a branchless binary search.
__device__ __forceinline__ int guard_pos(const float *row, float x) {
    int p = 0;
#pragma unroll
    for (int st = 32; st > 0; st >>= 1) p += row[p + st - 1] > x ? st : 0;
    return p;
}

// Sampled user r: one of the users r * stride .. r * stride + stride - 1, at a
// place that a hash of r gives.  A fixed place would fall into step with users
// stored in a periodic order (users of 16 clusters in turn, a stride of 15 or
// 16): 1000 queries over 1M such users overflowed their lists, 33 ms a call
// where this sample takes 1.25.  (r * stride < n_user < 2^31.)
__device__ __forceinline__ int64_t sample_user(int64_t r, int64_t stride, int64_t n_user) {
    uint32_t h = (uint32_t)r * 0x9E3779B1u;
    h = (h ^ (h >> 15)) * 0x85EBCA6Bu;
    return min((uint32_t)r * (uint32_t)stride + __umulhi(h, (uint32_t)stride), (uint32_t)n_user - 1u);
}

// Guard rows of NU sampled users (r0 + i, i < NU, clamped to the last) to LDS rows
// of stride GW + 1: an odd stride, so the lanes' searches fall in different banks.
// Every load is in flight before the first write.
constexpr int GP = GW + 1;
template <int NU>
__device__ __forceinline__ void stage_guards(float *dst, const float *__restrict__ gvals, int64_t r0, int64_t n_s,
                                             int64_t stride, int64_t n_user) {
    constexpr int N = NU * GW / 4 / NT;
    f32x4 v[N];
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const int c = (int)threadIdx.x + k * NT;
        v[k] = reinterpret_cast<const f32x4 *>(gvals)[
            sample_user(min(r0 + c / (GW / 4), n_s - 1), stride, n_user) * (GW / 4) + c % (GW / 4)];
    }
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const int c = (int)threadIdx.x + k * NT;
        float *d = dst + (c / (GW / 4)) * GP + c % (GW / 4) * 4;
#pragma unroll
        for (int j = 0; j < 4; ++j) d[j] = v[k][j];
    }
}

// A float below x (finite): below(a - b) <= the exact a - b.
__device__ __forceinline__ float below(float x) {
    const int32_t i = __float_as_int(x);
    return __int_as_float(x > 0.0f ? i - 1 : x < 0.0f ? i + 1 : (int32_t)0x80000001u);
}

// guard_pos with every eighth value of the row in registers: hd[j] = row[8 j + 7].
// Three steps there, three in LDS.
__device__ __forceinline__ int guard_pos_reg(const float (&hd)[7], const float *row, float x) {
    const bool b2 = hd[3] > x;
    const float h1 = __builtin_unpredictable(b2) ? hd[5] : hd[1];
    const bool b1 = h1 > x;
    const float ha = __builtin_unpredictable(b1) ? hd[6] : hd[4], hb = __builtin_unpredictable(b1) ? hd[2] : hd[0];
    const bool b0 = (__builtin_unpredictable(b2) ? ha : hb) > x;
    int p = (b2 ? 32 : 0) + (b1 ? 16 : 0) + (b0 ? 8 : 0);
#pragma unroll
    for (int st = 4; st > 0; st >>= 1) p += row[p + st - 1] > x ? st : 0;
    return p;
}

// ---- sample ----------------------------------------------------------------
// hist[b * 64 + p] += #{sampled users with p fine columns above s - e}, p <
// n_fine, and in the bits from kPossible up the same for s + e, from one pair in
// kPossibleOf: the first says which column enough users reach for certain, both
// together how many users the list at that column holds.  (With a search of its
// own for s + e in every pair the sample takes twice as long.)  A workgroup takes
// one stage of 64 queries (blockIdx.y) and every gridDim.x-th block of 128
// sampled users, so its counts leave LDS once.  Queries are the A operand, users
// the B operand: lane (lr, lq) of a 16 x 16 block owns user lr and queries
// 4 lq .. 4 lq + 3.  PROD: one product u_hi q_hi, or three with the low halves.
constexpr int kPossible = 18, kPossibleOf = 32;  // n_s < 2^17: 18 bits hold a certain count, 14 a possible one
template <int KS, int PROD>
__global__ void __launch_bounds__(NT, PROD == 1 && KS <= 7 ? 2 : 1) k_sample_screen(ListScreen P, int64_t n_s, int64_t stride,
                                                         int64_t n_user, uint32_t *__restrict__ hist) {
    constexpr int ROWQ = (KS * 32 + KPAD_LDS) / 8, KQ = KS * 4, NH = PROD == 1 ? 1 : 2;
    __shared__ u32x4 sA[NH][QST * ROWQ];
    __shared__ float sCs[QST];
    __shared__ float sG[128 * GP];
    __shared__ uint32_t sH[QST * GW];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lr = lane & 15, lq = lane >> 4;
    const int32_t q0 = (int32_t)blockIdx.y * QST;
#pragma unroll
    for (int h = 0; h < NH; ++h) {
        const u32x4 *src = reinterpret_cast<const u32x4 *>(h ? P.q_lo : P.q_hi);
        u32x4 pre[KS];
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            const int c = (int)threadIdx.x + k * NT;
            pre[k] = src[(int64_t)min(q0 + c / KQ, P.nq - 1) * KQ + c % KQ];
        }
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            const int c = (int)threadIdx.x + k * NT;
            sA[h][(c / KQ) * ROWQ + c % KQ] = pre[k];
        }
    }
    if (threadIdx.x < QST) sCs[threadIdx.x] = P.q_cs[min(q0 + (int)threadIdx.x, P.nq - 1)];
    for (int i = threadIdx.x; i < QST * GW; i += NT) sH[i] = 0u;
    const int64_t n_rb = (n_s + 127) / 128;
    uint32_t turn = blockIdx.x;  // which of a block's pairs are searched for s + e too
    for (int64_t rb = blockIdx.x; rb < n_rb; rb += gridDim.x, turn += gridDim.x + 1) {
        __syncthreads();  // the previous block is done with sG
        stage_guards<128>(sG, P.gvals, rb * 128, n_s, stride, n_user);
        Frag uh[2][KS], ul[PROD == 1 ? 1 : 2][PROD == 1 ? 1 : KS];
        float ar[2];
        bool live[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int64_t r = rb * 128 + wave * 32 + b * 16 + lr;
            live[b] = r < n_s;
            const int64_t u = sample_user(min(r, n_s - 1), stride, n_user);
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) uh[b][ks].q = reinterpret_cast<const u32x4 *>(P.user_hi + u * P.Kp)[ks * 4 + lq];
            if constexpr (PROD > 1)
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) ul[b][ks].q = reinterpret_cast<const u32x4 *>(P.user_lo + u * P.Kp)[ks * 4 + lq];
            ar[b] = P.C * P.user_norm[u];
        }
        __syncthreads();
        float hd[2][7];
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int j = 0; j < 7; ++j) hd[b][j] = sG[(wave * 32 + b * 16 + lr) * GP + 8 * j + 7];
#pragma unroll 1
        for (int g = 0; g < QST / 16 && q0 + g * 16 < P.nq; ++g) {
            f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                Frag qh;
                qh.q = sA[0][(g * 16 + lr) * ROWQ + ks * 4 + lq];
                [[maybe_unused]] Frag ql;
                if constexpr (PROD > 1) ql.q = sA[NH - 1][(g * 16 + lr) * ROWQ + ks * 4 + lq];
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qh.v, uh[b][ks].v, acc[b], 0, 0, 0);
                    if constexpr (PROD > 1) {
                        acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ql.v, uh[b][ks].v, acc[b], 0, 0, 0);
                        acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qh.v, ul[b][ks].v, acc[b], 0, 0, 0);
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int ql = g * 16 + 4 * lq + i;
                const float cs = sCs[ql];
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    const float e = __fmaf_rn(ar[b], cs, P.floor);
                    const float *row = &sG[(wave * 32 + b * 16 + lr) * GP];
                    const int p = guard_pos_reg(hd[b], row, acc[b][i] - e);
                    if (live[b] && p < P.n_fine) atomicAdd(&sH[ql * GW + p], 1u);
                }
            }
            if (g == (int)(turn & 3)) {  // uniform, as is the next: one search a block, so no workgroup has more
                static_assert(kPossibleOf == 4 * 8, "one of 8 pairs of one of 4 groups of queries");
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    if ((int)(turn >> 2 & 7) == j) {
                        const int b = j >> 2, ql = g * 16 + 4 * lq + (j & 3);
                        const float e = __fmaf_rn(ar[b], sCs[ql], P.floor);
                        const int p = guard_pos_reg(hd[b], &sG[(wave * 32 + b * 16 + lr) * GP], acc[b][j & 3] + e);
                        if (live[b] && p < P.n_fine) atomicAdd(&sH[ql * GW + p], 1u << kPossible);
                    }
            }
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < QST * GW; i += NT)
        if (sH[i] && q0 + i / GW < P.nq) atomicAdd(&hist[(int64_t)q0 * GW + i], sH[i]);
}

// The same counts from exact scores qip[b * n_user + u].
__global__ void __launch_bounds__(NT) k_sample_scores(const float *__restrict__ qip, int64_t n_user, int32_t nq, float eps,
                                                      const float *__restrict__ gvals, int32_t n_fine, int64_t n_s,
                                                      int64_t stride, uint32_t *__restrict__ hist, uint64_t *t) {
    stamp(t);
    constexpr int UB = 64, QB = 16;
    __shared__ float sG[UB * GP];
    __shared__ uint32_t sH[QB * GW];
    const int32_t q0 = (int32_t)blockIdx.y * QB;
    for (int i = threadIdx.x; i < QB * GW; i += NT) sH[i] = 0u;
    const int64_t n_ub = (n_s + UB - 1) / UB;
    for (int64_t ub = blockIdx.x; ub < n_ub; ub += gridDim.x) {
        __syncthreads();
        stage_guards<UB>(sG, gvals, ub * UB, n_s, stride, n_user);
        __syncthreads();
        const int ul = threadIdx.x & 63;
        const int64_t r = ub * UB + ul;
        const int64_t u = sample_user(min(r, n_s - 1), stride, n_user);
        if (r < n_s)
            for (int ql = threadIdx.x >> 6; ql < QB && q0 + ql < nq; ql += NT / 64) {
                const float s = qip[(int64_t)(q0 + ql) * n_user + u];
                const int p = guard_pos(&sG[ul * GP], eps > 0.0f ? __double2float_rd((double)s - (double)eps) : s);
                if (p < n_fine) atomicAdd(&sH[ql * GW + p], 1u);
            }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < QB * GW; i += NT)
        if (sH[i] && q0 + i / GW < nq) atomicAdd(&hist[(int64_t)q0 * GW + i], sH[i]);
}

// ---- plan ------------------------------------------------------------------
// One workgroup.  Each query's threshold column, the queries ordered by it
// (slot -> query), and for every four neighbouring slots the column they share,
// the largest of theirs (a larger column lists more users, never fewer).  A
// query with no such column, or with a list that the scores' error takes past
// cap, gets thr = -1 (finer scores answer it) and no slot, one whose list is over
// cap without the error kNoList (a search over every user answers it).  So do the
// queries whose lists the scores' error makes more than `band` pairs longer, and
// those whose lists are longer than `share`, if that is enough in all to pay for
// what another attempt costs however few its queries: kBandMin pairs, the 80 us
// of a pass from finer scores, or kSearchUsers pairs a user, the search's 4 ms at
// 1M users (nothing if some query is searched anyway).  Lists are taken in order of
// their length, up to `room` pairs; the longer ones get thr = kNoRoom and
// ctr->n_need says how many pairs they hold.  (Taken in order of their column,
// popular queries came first and one of them kept every other out.)
// Four slots of different columns are estimated again at the shared one: a query
// that few users rank high can make three others list most users.  Where such a
// list is over cap, or what all of them add does not fit the arrays and the four
// take more than an equal share of what is left of them, they keep a smaller one
// of their columns and the deeper queries get thr = kNoRoom.
constexpr int PT = 1024;
constexpr int64_t kBandMin = 400000, kSearchUsers = 12;

__global__ void __launch_bounds__(PT) k_list_plan(const uint32_t *__restrict__ hist, int32_t nq, int32_t n_fine,
                                                  int64_t stride, int64_t n_user, int64_t cap, int64_t share,
                                                  int64_t band, int64_t room, int64_t list_cap,
                                                  uint64_t coarse_mask, QueryInfo *__restrict__ qi,
                                                  int32_t *__restrict__ order, int32_t *__restrict__ colg,
                                                  ListCounters *__restrict__ ctr) {
    __shared__ int32_t bin[GW], at[GW], mix[GW];
    __shared__ int64_t load[GW];  // pairs of the lists of each length class
    __shared__ int64_t longer[2];  // pairs that the scores' error adds to lists it makes `band` longer; past `share`
    __shared__ int64_t left, added;  // room beside the lists at their own columns, and what sharing adds
    __shared__ int32_t n_finer, n_slots, n_mix, longest, searched;
    // pairs of a list that `certain` sampled users reach for certain, and so many
    // of the few searched for it possibly
    constexpr uint32_t kCertain = (1u << kPossible) - 1;
    auto estimate = [&](int64_t certain, int64_t possible) {
        return min(max(certain, possible * kPossibleOf) * stride, n_user);
    };
    // two length classes an octave
    auto length_class = [](int32_t n) {
        const int top = 31 - __clz(max(n, 1));
        return 2 * top + (top > 0 ? n >> (top - 1) & 1 : 0);
    };
    // the columns' first slots: a column per lane of one wavefront
    auto first_slots = [&] {
        const int t = threadIdx.x;
        const int32_t own = bin[t];
        int32_t s = own;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int32_t z = __shfl_up(s, o, 64);
            if (t >= o) s += z;
        }
        const int32_t first = s - own;
        at[t] = first;
        bin[t] = 0;
        // the groups of four that hold more than one column, at the first of
        // the columns that start inside them
        const uint64_t in = __builtin_amdgcn_ballot_w64(own > 0 && first % 4 != 0);
        const uint64_t before = in & ((1ull << t) - 1);
        const int32_t prev = __shfl(first, before ? 63 - __clzll((long long)before) : 0, 64);
        mix[t] = ((in >> t) & 1) && (!before || prev / 4 != first / 4) ? first / 4 : -1;
        const int groups = (int)__popcll(__builtin_amdgcn_ballot_w64(mix[t] >= 0));
        if (t == 63) {
            n_slots = s;
            n_mix = groups;
        }
    };
    auto column_of = [&](int32_t slot) {  // the last column that starts at or before it
        int t = 0;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) t += at[t + o] <= slot ? o : 0;
        return t;
    };
    for (int i = threadIdx.x; i < GW; i += PT) { bin[i] = 0; load[i] = 0; }
    if (threadIdx.x == 0) n_finer = n_slots = n_mix = longest = searched = 0, longer[0] = longer[1] = left = added = 0;
    __syncthreads();
    int32_t own_thr = -1;  // of the thread's first query, which then needs no reading back
    for (int32_t b = threadIdx.x; b < nq; b += PT) {
        // the row's 64 counts in flight together (read one after the other, the
        // early end of the search costs more than it saves)
        u32x4 v[GW / 4];
#pragma unroll
        for (int j = 0; j < GW / 4; ++j) v[j] = reinterpret_cast<const u32x4 *>(hist + (int64_t)b * GW)[j];
        const int32_t k = qi[b].topk;
        const double mean = (double)k / (double)stride;
        const uint32_t want = stride == 1 ? (uint32_t)k : (uint32_t)(mean + 3.0 * sqrt(mean) + 4.0) + 1u;
        // the sums grow with the column: the first one that reaches `want` is the
        // smallest that does (there are none past the fine columns)
        int32_t t = 0;
        uint32_t cum = 0, pos = 0, certain = ~0u, possible = ~0u;
#pragma unroll
        for (int f = 0; f < GW; ++f) {
            cum += v[f / 4][f % 4] & kCertain;
            pos += v[f / 4][f % 4] >> kPossible;
            t += cum < want ? 1 : 0;
            certain = min(certain, cum < want ? ~0u : cum);
            possible = min(possible, cum < want ? ~0u : pos);
        }
        if (t >= n_fine) { t = -1; certain = possible = 0; }
        const int64_t n = estimate(certain, possible);
        const int64_t error = n - min(certain * stride, n_user);
        if (n - error > cap) {
            t = kNoList;
            searched = 1;
        } else if (n > cap && 4 * error > n) {
            t = -1;
        }
        if (b < PT) own_thr = t;
        qi[b].thr = t;
        qi[b].n_cand = (int32_t)n;  // until the candidates are counted
        qi[b].n_dropped = (int32_t)error;
        if (t >= 0) {
            if (error > band) atomicAdd(reinterpret_cast<unsigned long long *>(&longer[0]), (unsigned long long)error);
            if (n > share) atomicAdd(reinterpret_cast<unsigned long long *>(&longer[1]), (unsigned long long)(n - share));
            atomicAdd(&bin[t], 1);
            atomicAdd(reinterpret_cast<unsigned long long *>(&load[length_class((int32_t)n)]), (unsigned long long)n);
        }
    }
    __syncthreads();
    const bool by_band = longer[0] > kBandMin, by_length = longer[1] > (searched ? 0 : kSearchUsers * n_user);
    if (by_band || by_length) {  // uniform
        for (int i = threadIdx.x; i < GW; i += PT) { bin[i] = 0; load[i] = 0; }
        __syncthreads();
        for (int32_t b = threadIdx.x; b < nq; b += PT) {
            const int32_t t = qi[b].thr;
            if (t < 0) continue;
            if ((by_band && qi[b].n_dropped > band) || (by_length && qi[b].n_cand > share)) {
                const int32_t why = by_band && qi[b].n_dropped > band ? -1 : kNoList;
                qi[b].thr = why;
                if (b < PT) own_thr = why;
                continue;
            }
            atomicAdd(&bin[t], 1);
            atomicAdd(reinterpret_cast<unsigned long long *>(&load[length_class(qi[b].n_cand)]), (unsigned long long)qi[b].n_cand);
        }
        __syncthreads();
    }
    static_assert(GW == 64, "one wavefront");
    if (threadIdx.x < 64) {
        const int t = threadIdx.x;
        int64_t sum = load[t];
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int64_t y = __shfl_up(sum, o, 64);
            if (t >= o) sum += y;
        }
        const uint64_t m = __builtin_amdgcn_ballot_w64(sum <= room);  // loads are not negative: true up to some class
        const int last = m ? 63 - __clzll((long long)m) : -1;
        const int64_t all = __shfl(sum, 63, 64), in = last >= 0 ? __shfl(sum, max(last, 0), 64) : 0;
        if (t == 0) {
            longest = last;
            left = list_cap / 8 * 7 - in;
            ctr->n_need = (unsigned long long)(all - in);
        }
        if (last == 63) first_slots();
        else bin[t] = 0;
    }
    __syncthreads();
    if (longest < 63) {  // uniform: some lists find no room
        for (int32_t b = threadIdx.x; b < nq; b += PT) {
            const int32_t t = qi[b].thr;
            if (t < 0) continue;
            if (length_class(qi[b].n_cand) <= longest) {
                atomicAdd(&bin[t], 1);
            } else {
                qi[b].thr = kNoRoom;
                if (b < PT) own_thr = kNoRoom;
            }
        }
        __syncthreads();
        if (threadIdx.x < 64) first_slots();
        __syncthreads();
    }
    for (int32_t b = threadIdx.x; b < nq; b += PT) {
        const int32_t t = b < PT ? own_thr : qi[b].thr;
        if (t < 0) continue;
        order[at[t] + atomicAdd(&bin[t], 1)] = b;
        if (!((coarse_mask >> t) & 1)) atomicAdd(&n_finer, 1);
    }
    __threadfence_block();
    __syncthreads();
    for (int32_t g = threadIdx.x; g < (n_slots + 3) / 4; g += PT) {
        const int32_t c = column_of(4 * g);
        if (column_of(min(4 * g + 3, n_slots - 1)) == c) colg[g] = c;
    }
    // a thread per member of the mixed groups
    const int32_t g = threadIdx.x < 4 * GW ? mix[threadIdx.x >> 2] : -1;
    const int32_t slot = 4 * g + (int32_t)(threadIdx.x & 3);
    const bool member = g >= 0 && slot < n_slots;
    const int32_t b = member ? order[slot] : 0;
    const int32_t own = member ? column_of(slot) : -1;
    // the group's columns: the largest, the next one below it, the smallest
    auto quad_max = [](int32_t x) {
        x = max(x, __shfl_xor(x, 1, 64));
        return max(x, __shfl_xor(x, 2, 64));
    };
    const int32_t c0 = quad_max(own), c1 = quad_max(own < c0 ? own : -1);
    const int32_t least = __shfl(own, (int)(threadIdx.x & 63 & ~3), 64);
    int64_t more[2] = {0, 0};
    bool over[2] = {false, false};
    if (member && own < c0) {
        const u32x4 *row = reinterpret_cast<const u32x4 *>(hist + (int64_t)b * GW);
        uint32_t cum[2] = {0, 0}, pos[2] = {0, 0};
#pragma unroll
        for (int j = 0; j < GW / 4; ++j) {
            const u32x4 v = row[j];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t x0 = 4 * j + i <= c0 ? v[i] : 0u, x1 = 4 * j + i <= c1 ? v[i] : 0u;
                cum[0] += x0 & kCertain;
                pos[0] += x0 >> kPossible;
                cum[1] += x1 & kCertain;
                pos[1] += x1 >> kPossible;
            }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int64_t n = estimate(cum[h], pos[h]);
            more[h] = n - qi[b].n_cand;
            over[h] = n > cap;
        }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        more[h] += __shfl_xor(more[h], 1, 64);
        more[h] += __shfl_xor(more[h], 2, 64);
        over[h] = (__builtin_amdgcn_ballot_w64(over[h]) >> (threadIdx.x & 63 & ~3) & 0xF) != 0;
    }
    if (g >= 0 && (threadIdx.x & 3) == 0)
        atomicAdd(reinterpret_cast<unsigned long long *>(&added), (unsigned long long)more[0]);
    __syncthreads();
    if (member) {
        auto good = [&](int h) { return !over[h] && more[h] <= left / n_mix; };
        const int32_t c = !over[0] && added <= left ? c0 : good(0) ? c0 : good(1) ? c1 : least;
        qi[b].thr = own <= c ? c : kNoRoom;
        if ((threadIdx.x & 3) == 0) colg[g] = c;
    }
    if (threadIdx.x == 0) {
        ctr->n_slots = n_slots;
        ctr->n_finer = n_finer;
    }
}

// ---- list ------------------------------------------------------------------
// The list's length as every later stage reads it: none of a list that outgrew
// its arrays.  Its pairs are not all there, and in a batch that orders them by
// query the ordered arrays are never written, so no stage may walk them.
__device__ __forceinline__ int64_t list_len(const ListCounters *ctr, int64_t cap) {
    const int64_t n = (int64_t)ctr->n_list;
    return n <= cap ? n : 0;
}

// n places of the list, counted in 64 bits; past the list's capacity its end (32
// bits hold it, cap <= INT32_MAX / 2), where nothing is written.
__device__ __forceinline__ int32_t list_places(unsigned long long *list_n, int32_t n, int64_t cap) {
    const unsigned long long first = atomicAdd(list_n, (unsigned long long)n);
    return (int32_t)min(first, (unsigned long long)cap);
}

// Zeroes the list's counts per query and the scatter's cursors behind them.
__device__ __forceinline__ void zero_counts(int32_t nq, uint32_t *__restrict__ g_cnt) {
    if (g_cnt && blockIdx.y == 0)
        for (int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x; i < 2 * (int64_t)nq; i += (int64_t)gridDim.x * NT) g_cnt[i] = 0u;
}

constexpr int QCAP = 512;    // listed pairs of a unit queued in LDS
// slots per unit of k_list_screen: a unit's user rows are read once per slice,
// and its workgroup runs long enough to hide them
constexpr int kSlice = 512;

struct ListQueue {
    uint2 e[QCAP];
    int32_t n, base;
};

// Appends each lane's pairs (bit 4 b + i of m: user u0 + 16 b, query slot_b[i])
// to the queue, or, where it is full, to the list, with one atomic per
// wavefront.  Called by whole wavefronts.
__device__ __forceinline__ void list_put(ListQueue &sq, uint32_t m, int32_t u0, const int32_t *slot_b,
                                         int32_t *__restrict__ cl_u, int32_t *__restrict__ cl_b, int64_t cap,
                                         unsigned long long *__restrict__ list_n) {
    const int lane = threadIdx.x & 63;
    const int32_t c = __popc(m);
    int32_t x = c;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    const int32_t tot = __shfl(x, 63, 64);
    int32_t base = 0;
    if (lane == 0) base = atomicAdd(&sq.n, tot);
    base = __shfl(base, 0, 64);
    int32_t p = base + x - c;
    // places at and past QCAP: the wavefront's share of the list
    int32_t over = 0;
    if (base + tot > QCAP) {
        const int32_t first = max(base, QCAP);
        if (lane == 0) over = list_places(list_n, base + tot - first, cap);
        over = __shfl(over, 0, 64) - first;
    }
    while (m) {
        const int t = __ffs(m) - 1;
        m &= m - 1;
        const int32_t u = u0 + (t >> 2) * 16, b = slot_b[t & 3];
        if (p < QCAP) {
            sq.e[p] = make_uint2((uint32_t)u, (uint32_t)b);
        } else if ((int64_t)over + p < cap) {
            cl_u[over + p] = u;
            cl_b[over + p] = b;
        }
        ++p;
    }
}

// The unit's queued pairs go to the list; every wave has passed a barrier
// since the last push, and passes one before the next.
__device__ __forceinline__ void list_flush(ListQueue &sq, int32_t *__restrict__ cl_u, int32_t *__restrict__ cl_b,
                                           int64_t cap, unsigned long long *__restrict__ list_n) {
    const int32_t n = min(sq.n, QCAP);
    if (n > 0) {  // uniform
        if (threadIdx.x == 0) sq.base = list_places(list_n, n, cap);
        __syncthreads();
        const int64_t base = sq.base;
        for (int i = threadIdx.x; i < n; i += NT)
            if (base + i < cap) { cl_u[base + i] = (int32_t)sq.e[i].x; cl_b[base + i] = (int32_t)sq.e[i].y; }
        __syncthreads();
        if (threadIdx.x == 0) sq.n = 0;
    }
}

// A wavefront's listed pairs, user in the unit | slot in the slice << 8, and
// their number in a register of every lane.
constexpr int WQ = 256;

__device__ __forceinline__ void wave_flush(const uint32_t *q, int n, int32_t base, int32_t u0, const int32_t *ord,
                                           int32_t *__restrict__ cl_u, int32_t *__restrict__ cl_b, int64_t cap) {
    for (int i = threadIdx.x & 63; i < n; i += 64)
        if ((int64_t)base + i < cap) {
            cl_u[base + i] = u0 + (int32_t)(q[i] & 0xFFu);
            cl_b[base + i] = ord[q[i] >> 8];
        }
}

// Lists from the matrix cores.  Unit = 64 NB users (each wave 16 NB, held in
// VGPRs) x a slice of the slots, 64 queries at a time through LDS (two buffers:
// the next stage's rows go straight to LDS while one is computed, one barrier
// per stage); a block's thresholds are loaded while the previous one is
// computed.  With PROD = 3 the stage is 32 queries' hi and lo rows.  A
// workgroup whose pairs find the list full stops there (reading the counter at
// the start of each unit instead took 140 of 705 us, 1M users x 1000 queries).
// A pair costs one fused multiply-add and one compare beside its share of the
// matrix products; listed pairs are queued per wavefront without an atomic, and
// a unit takes its part of the list with one.  Bound: the matrix cores' 16
// cycles per 16x16x32 product and about 100 VALU instructions per 16 queries x
// 16 NB users beside them: 573 us at 1M users x 150 dims x 1000 queries, 560
// TFLOP/s (80 bytes a thread spilled).
template <int KS, int NB, int PROD>
__global__ void __launch_bounds__(NT, PROD == 1 && KS <= 5 ? 3 : 2) k_list_screen(ListScreen P, int64_t n_user,
                                                                     const int32_t *__restrict__ order,
                                                                     const int32_t *__restrict__ colg,
                                                                     uint32_t *__restrict__ g_cnt,
                                                                     ListCounters *__restrict__ ctr,
                                                                     int32_t *__restrict__ cl_u,
                                                                     int32_t *__restrict__ cl_b, int64_t list_cap) {
    constexpr int KQ = KS * 4, UB = 64 * NB, NH = PROD == 1 ? 1 : 2, QS = QST / NH;  // queries per stage
    static_assert(NH * QS * KQ == KS * NT, "KS 16-byte pieces per thread and stage");
    static_assert(UB <= 256 && kSlice % QST == 0, "a queued pair's user takes 8 bits");
    // two variables, not one array: a read of one then does not wait for the
    // loads into the other
    __shared__ u32x4 sA0[NH * QS * KQ], sA1[NH * QS * KQ];
    __shared__ f32x4 sCs[kSlice / 4];
    __shared__ int32_t sCol[kSlice / 4 + QST / 4], sOrd[kSlice];
    __shared__ uint32_t sQ[NT / 64][WQ];
    __shared__ int32_t sN[NT / 64], sBase;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lr = lane & 15, lq = lane >> 4;
    const int32_t n_slots = ctr->n_slots;
    zero_counts(P.nq, g_cnt);
    const int64_t n_rb = (n_user + UB - 1) / UB;
    const int64_t n_sl = (n_slots + kSlice - 1) / kSlice, n_units = n_rb * n_sl;
    for (int64_t unit = blockIdx.x; unit < n_units; unit += gridDim.x) {
        const int64_t rb = unit / n_sl;
        const int32_t s0 = (int32_t)(unit % n_sl) * kSlice, ns = min(n_slots - s0, kSlice);
        // the slice's queries, scales and threshold columns (slots past it repeat its last)
        for (int i = threadIdx.x; i < kSlice; i += NT) {
            const int32_t q = order[s0 + min(i, ns - 1)];
            sOrd[i] = q;
            reinterpret_cast<float *>(sCs)[i] = P.q_cs[q];
        }
        for (int i = threadIdx.x; i < kSlice / 4 + QST / 4; i += NT) sCol[i] = colg[(s0 + min(4 * i, ns - 1)) / 4];
        // the unit's rows: uniform base pointers and 32-bit offsets
        const int last = (int)min((int64_t)(UB - 1), n_user - 1 - rb * UB);
        const u32x4 *ubase = reinterpret_cast<const u32x4 *>(P.user_hi + rb * UB * P.Kp);
        const float *gbase = P.gcols + rb * UB, *nbase = P.user_norm + rb * UB;
        Frag uh[NB][KS], ul[PROD == 1 ? 1 : NB][PROD == 1 ? 1 : KS];
        float ar[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int at = wave * 16 * NB + b * 16 + lr, uc = min(at, last);
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) uh[b][ks].q = ubase[uc * KQ + ks * 4 + lq];
            if constexpr (PROD > 1) {
                const u32x4 *lbase = reinterpret_cast<const u32x4 *>(P.user_lo + rb * UB * P.Kp);
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) ul[b][ks].q = lbase[uc * KQ + ks * 4 + lq];
            }
            // rows past the last user never reach a threshold
            ar[b] = at <= last ? P.C * nbase[uc] : -INFINITY;
        }
        int n_q = 0;  // queued pairs of the wavefront
        auto load_stage = [&](u32x4 *dst, int32_t q) __attribute__((always_inline)) {  // slots s0 + q ..
#pragma unroll
            for (int k = 0; k < KS; ++k) {
                const int c = (int)threadIdx.x + k * NT, r = c / KQ % QS;
                const uint16_t *src = NH > 1 && c >= QS * KQ ? P.q_lo : P.q_hi;  // the same in a wavefront
                load_to_lds(reinterpret_cast<const u32x4 *>(src) + ((uint32_t)sOrd[q + r] * KQ + swizzled<KS>(r, c % KQ)),
                            dst + wave * 64 + k * NT);
            }
        };
        auto load_thr = [&](int32_t col, float (&t)[NB]) {
#pragma unroll
            for (int b = 0; b < NB; ++b) t[b] = gbase[(int64_t)col * P.pitch + min(wave * 16 * NB + b * 16 + lr, last)];
        };
        __syncthreads();  // sOrd, sCs and sCol are complete
        load_stage(sA0, 0);
        int32_t cur = sCol[lq];  // the lane's threshold column
        float raw[NB], thr[NB];
        load_thr(cur, raw);
        bool fresh = true;       // raw holds new thresholds (uniform)
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's rows are in LDS
        __syncthreads();
        auto stage = [&](const u32x4 *rows, u32x4 *ahead, int32_t q0) __attribute__((always_inline)) {
            if (q0 + QS < ns) load_stage(ahead, q0 + QS);
            const int n_g = min(QS / 16, (ns - q0 + 15) / 16);
#pragma unroll 1
            for (int g = 0; g < n_g; ++g) {
                const int t4 = (q0 >> 2) + g * 4 + lq;  // the lane's four slots: s0 + 4 t4 ..
                if (fresh) {
                    // s^ + e >= G with the floor taken off G, rounded down (one
                    // step below the rounded difference is below the difference)
#pragma unroll
                    for (int b = 0; b < NB; ++b) thr[b] = below(raw[b] - P.floor);
                }
                const int32_t next = sCol[t4 + 4];
                fresh = __builtin_amdgcn_ballot_w64(next != cur) != 0;
                if (fresh) {
                    cur = next;
                    load_thr(cur, raw);
                }
                f32x4 acc[NB];
#pragma unroll
                for (int b = 0; b < NB; ++b) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    Frag qh;
                    qh.q = rows[(g * 16 + lr) * KQ + swizzled<KS>(g * 16 + lr, ks * 4 + lq)];
#pragma unroll
                    for (int b = 0; b < NB; ++b)
                        acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qh.v, uh[b][ks].v, acc[b], 0, 0, 0);
                    if constexpr (PROD > 1) {
                        Frag ql;
                        ql.q = rows[QS * KQ + (g * 16 + lr) * KQ + swizzled<KS>(g * 16 + lr, ks * 4 + lq)];
#pragma unroll
                        for (int b = 0; b < NB; ++b) {
                            acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ql.v, uh[b][ks].v, acc[b], 0, 0, 0);
                            acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qh.v, ul[b][ks].v, acc[b], 0, 0, 0);
                        }
                    }
                }
                // D[4 lq + i][lr]: slot s0 + 4 t4 + i, user b * 16 + lr of the wave
                const f32x4 cs = sCs[t4];
                bool any = false;
#pragma unroll
                for (int b = 0; b < NB; ++b)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        acc[b][i] = __fmaf_rn(ar[b], cs[i], acc[b][i]);
                        any |= acc[b][i] >= thr[b];
                    }
                if (__builtin_amdgcn_ballot_w64(any) != 0) {
#pragma unroll
                    for (int b = 0; b < NB; ++b)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const bool hit = acc[b][i] >= thr[b] && 4 * t4 + i < ns;
                            const uint64_t m = __builtin_amdgcn_ballot_w64(hit);
                            if (m != 0) {
                                if (n_q + 64 > WQ) {  // uniform: make room
                                    int32_t base = 0;
                                    if (lane == 0) base = list_places(&ctr->n_list, n_q, list_cap);
                                    wave_flush(sQ[wave], n_q, __shfl(base, 0, 64), (int32_t)(rb * UB), sOrd, cl_u, cl_b,
                                               list_cap);
                                    n_q = 0;
                                }
                                const int at = n_q + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                                                    __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
                                if (hit) sQ[wave][at] = (uint32_t)(wave * 16 * NB + b * 16 + lr) | (uint32_t)(4 * t4 + i) << 8;
                                n_q += (int)__popcll(m);
                            }
                        }
                }
            }
            __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's rows of the next stage are in LDS
            __syncthreads();
        };
        for (int32_t q0 = 0; q0 < ns; q0 += 2 * QS) {
            stage(sA0, sA1, q0);
            if (q0 + QS < ns) stage(sA1, sA0, q0 + QS);
        }
        // the unit's pairs: one place in the list for the four wavefronts
        if (lane == 0) sN[wave] = n_q;
        __syncthreads();
        int32_t before = 0, tot = 0;
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) {
            before += w < wave ? sN[w] : 0;
            tot += sN[w];
        }
        if (tot > 0) {  // uniform
            if (threadIdx.x == 0) sBase = list_places(&ctr->n_list, tot, list_cap);
            __syncthreads();
            const int32_t base = sBase;
            if (base >= list_cap) return;  // uniform: the list has outgrown its arrays, no stage will read it
            wave_flush(sQ[wave], n_q, base + before, (int32_t)(rb * UB), sOrd, cl_u, cl_b, list_cap);
        }
        __syncthreads();  // the next unit rewrites the slice, the queues and the stages
    }
}

// Lists from exact scores: one thread per user and a slice of the slots
// (blockIdx.y), four slots of one threshold column at a time; scores and
// thresholds are read in whole lines per wavefront.
constexpr int kScoreSlice = 64;

__global__ void __launch_bounds__(NT) k_list_scores(const float *__restrict__ qip, int64_t n_user, float eps,
                                                    const float *__restrict__ gcols, int64_t pitch,
                                                    const int32_t *__restrict__ order, const int32_t *__restrict__ colg,
                                                    int32_t nq, uint32_t *__restrict__ g_cnt,
                                                    ListCounters *__restrict__ ctr, int32_t *__restrict__ cl_u,
                                                    int32_t *__restrict__ cl_b, int64_t list_cap) {
    __shared__ ListQueue sq;
    __shared__ int32_t sB[kScoreSlice], sCol[kScoreSlice / 4];
    const int32_t n_slots = ctr->n_slots;
    zero_counts(nq, g_cnt);
    const int32_t s0 = (int32_t)blockIdx.y * kScoreSlice, ns = min(n_slots - s0, kScoreSlice);
    if (ns <= 0) return;
    if (threadIdx.x == 0) sq.n = 0;
    if (threadIdx.x < kScoreSlice) sB[threadIdx.x] = order[s0 + min((int)threadIdx.x, ns - 1)];
    if (threadIdx.x < kScoreSlice / 4) sCol[threadIdx.x] = colg[(s0 + min(4 * (int)threadIdx.x, ns - 1)) / 4];
    __syncthreads();
    const int64_t u = (int64_t)blockIdx.x * NT + threadIdx.x, uc = min(u, n_user - 1);
    for (int32_t s = 0; s < ns; s += 8) {
        float x[8], thr[2];
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = qip[(int64_t)sB[s + j] * n_user + uc];
#pragma unroll
        for (int j = 0; j < 2; ++j) thr[j] = gcols[(int64_t)sCol[s / 4 + j] * pitch + uc];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            uint32_t m = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float v = x[4 * j + i], hi = eps > 0.0f ? __double2float_ru((double)v + (double)eps) : v;
                m |= hi >= thr[j] && u < n_user && s + 4 * j + i < ns ? 1u << i : 0u;
            }
            if (__builtin_amdgcn_ballot_w64(m != 0) != 0)
                list_put(sq, m, (int32_t)u, &sB[s + 4 * j], cl_u, cl_b, list_cap, &ctr->n_list);
        }
    }
    __syncthreads();
    list_flush(sq, cl_u, cl_b, list_cap, &ctr->n_list);
}

// ---- the listed pairs by query ------------------------------------------------
// Batches of more than kFilterQueries queries have their list ordered by query:
// pairs per query, their places, and the pairs moved there.  The k-th bound and
// the candidates then are one workgroup's work per query, in LDS.  (With counts
// and places by global atomics per pair, the adds to one query's counter follow
// one another: with queries that 100k users rank first, 3.8M pairs of 1024 queries,
// the exact stage took 2.2 ms and the candidates' 0.9; now 0.54 and 0.30, and
// 0.18 for the order.)
// One contiguous chunk of the list per workgroup, counted in LDS, so a query
// takes one global add per chunk.
constexpr int CT = 1024;
constexpr int kGroupQ = 4096;       // queries counted in LDS at a time
constexpr int64_t kChunk = 1024;    // pairs of a workgroup, at least

__device__ __forceinline__ bool list_chunk(const ListCounters *ctr, int64_t cap, int64_t &first, int64_t &last) {
    const int64_t n = list_len(ctr, cap);
    const int64_t per = max(kChunk, (n + gridDim.x - 1) / gridDim.x);
    first = min(n, (int64_t)blockIdx.x * per);
    last = min(n, first + per);
    return first < last;
}

__device__ __forceinline__ void count_queries(uint32_t *h, const int32_t *__restrict__ raw_b, int64_t first,
                                              int64_t last, int32_t q0) {
    for (int j = threadIdx.x; j < kGroupQ; j += CT) h[j] = 0u;
    __syncthreads();
    for (int64_t i = first + threadIdx.x; i < last; i += CT) {
        const uint32_t j = (uint32_t)(raw_b[i] - q0);
        if (j < (uint32_t)kGroupQ) atomicAdd(&h[j], 1u);
    }
    __syncthreads();
}

// Pairs per query.
__global__ void __launch_bounds__(CT) k_list_count(const int32_t *__restrict__ raw_b, int64_t cap, int32_t nq,
                                                   uint32_t *__restrict__ g_cnt, const ListCounters *__restrict__ ctr,
                                                   uint64_t *t) {
    stamp(t);
    __shared__ uint32_t h[kGroupQ];
    int64_t first, last;
    if (!list_chunk(ctr, cap, first, last)) return;
    for (int32_t q0 = 0; q0 < nq; q0 += kGroupQ) {
        count_queries(h, raw_b, first, last, q0);
        for (int j = threadIdx.x; j < kGroupQ; j += CT)
            if (h[j]) atomicAdd(&g_cnt[q0 + j], h[j]);
        __syncthreads();
    }
}

// Every workgroup sums the counts to places itself (a last workgroup that does
// it for all needs a device-wide fence per workgroup: 36 us for 64 queries,
// where the count takes 5), the first one writes them for the candidates.
__global__ void __launch_bounds__(CT) k_list_scatter(const int32_t *__restrict__ raw_u, const int32_t *__restrict__ raw_b,
                                                     int64_t cap, int32_t nq, const uint32_t *__restrict__ g_cnt,
                                                     uint32_t *__restrict__ g_off, uint32_t *__restrict__ g_cur,
                                                     const ListCounters *__restrict__ ctr, int32_t *__restrict__ cl_u,
                                                     int32_t *__restrict__ cl_b) {
    constexpr int PER = kGroupQ / CT;
    __shared__ uint32_t h[kGroupQ], red[CT / 64];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    int64_t first, last;
    const bool work = list_chunk(ctr, cap, first, last);
    if (!work && blockIdx.x != 0) return;
    uint32_t before = 0;
    for (int32_t q0 = 0; q0 < nq; q0 += kGroupQ) {
        count_queries(h, raw_b, first, last, q0);
        // the thread's PER queries: places of the query and, in it, of the chunk
        const int32_t j0 = (int32_t)threadIdx.x * PER;
        uint32_t v[PER], own = 0;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            v[i] = q0 + j0 + i < nq ? g_cnt[q0 + j0 + i] : 0u;
            own += v[i];
        }
        uint32_t x = own;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(x, o, 64);
            if (lane >= o) x += y;
        }
        if (lane == 63) red[w] = x;
        __syncthreads();
        uint32_t base = before + x - own;
        for (int i = 0; i < CT / 64; ++i) {
            base += i < w ? red[i] : 0u;
            before += red[i];
        }
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int32_t j = j0 + i;
            if (blockIdx.x == 0 && q0 + j < nq) g_off[q0 + j] = base;
            if (h[j]) h[j] = base + atomicAdd(&g_cur[q0 + j], h[j]);
            base += v[i];
        }
        __syncthreads();
        for (int64_t i = first + threadIdx.x; i < last; i += CT) {
            const int32_t b = raw_b[i];
            const uint32_t j = (uint32_t)(b - q0);
            if (j >= (uint32_t)kGroupQ) continue;
            const uint32_t at = atomicAdd(&h[j], 1u);
            cl_u[at] = raw_u[i];
            cl_b[at] = b;
        }
        __syncthreads();
    }
}

// ---- exact scores, buckets and the k-th bound of the listed pairs -----------

// Workgroups are dispatched to the 8 XCDs in turn (block p on XCD p % 8), and
// each XCD has its own L2.  Block p takes logical block (p % 8) * per + p / 8 of
// the list, so each XCD takes one contiguous eighth of it: a unit's pairs (the
// same users) share one L2.  -1 past the list.
__device__ __forceinline__ int64_t xcd_block(int64_t n) {
    const int64_t blocks = (n + NT - 1) / NT, per = (blocks + 7) / 8;
    const int64_t p = blockIdx.x;
    if (p >= per * 8) return -1;
    const int64_t lb = (p % 8) * per + p / 8;
    return lb < blocks ? lb : -1;
}

// #{row[j] > x} when it is known to lie in [lo, hi].
__device__ __forceinline__ int32_t bucket_in(const float *__restrict__ row, int32_t lo, int32_t hi, float x) {
    while (lo < hi) {
        const int32_t mid = (lo + hi) >> 1;
        if (row[mid] > x) lo = mid + 1; else hi = mid;
    }
    return lo;
}

// #{T > x} of a user: the guard row's search (two cache lines) leaves the few
// columns between two fine columns.
__device__ __forceinline__ int32_t bucket_of(const float *__restrict__ grow, const float *__restrict__ row,
                                             const int32_t *col, int32_t n_fine, int32_t S, float x) {
    const int f = guard_pos(grow, x);
    return bucket_in(row, f > 0 ? col[f - 1] + 1 : 0, f < n_fine ? col[f] : S, x);
}

// The score rule's <u, q> of the 64 pairs of a wavefront, a pair per lane.  A
// lane that reads its own two rows touches a cache line of its own with every
// load, 64 lines per instruction; here the rows are read 64 bytes by four
// neighbouring lanes, 16 rows per instruction, and pass through the
// wavefront's LDS (rows of 16 terms and 4 floats of padding, so the 16-byte
// reads spread over all banks), 16 terms ahead of the sum.
constexpr int DC = 16, DP = DC + 4;

__device__ __forceinline__ float wave_rule_dot(f32x4 *su, f32x4 *sv, const float *__restrict__ users,
                                               const float *__restrict__ queries, int64_t u, int64_t b, int32_t ld,
                                               int32_t dim) {
    const int lane = threadIdx.x & 63, piece = lane & 3;
    const float *ru[4], *rq[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {  // rows 16 j + lane / 4 of the wavefront
        ru[j] = users + (int64_t)__shfl((int32_t)u, 16 * j + (lane >> 2), 64) * ld;
        rq[j] = queries + (int64_t)__shfl((int32_t)b, 16 * j + (lane >> 2), 64) * ld;
    }
    f32x4 xu[4], xq[4];
    auto load = [&](int32_t k0) {
        const int32_t k = min(k0 + 4 * piece, ld - 4);  // past the row's end: unused
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            xu[j] = *reinterpret_cast<const f32x4 *>(ru[j] + k);
            xq[j] = *reinterpret_cast<const f32x4 *>(rq[j] + k);
        }
    };
    load(0);
    float s = 0.0f;
    for (int32_t k0 = 0; k0 < dim; k0 += DC) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            su[(16 * j + (lane >> 2)) * (DP / 4) + piece] = xu[j];
            sv[(16 * j + (lane >> 2)) * (DP / 4) + piece] = xq[j];
        }
        if (k0 + DC < dim) load(k0 + DC);
        // this wavefront's LDS only, whose operations are in order
        __builtin_amdgcn_wave_barrier();
        const int32_t n = min(DC, dim - k0);
        f32x4 a[DC / 4], c[DC / 4];
#pragma unroll
        for (int j = 0; j < DC / 4; ++j) {
            a[j] = su[lane * (DP / 4) + j];
            c[j] = sv[lane * (DP / 4) + j];
        }
        __builtin_amdgcn_wave_barrier();
        if (n == DC) {
#pragma unroll
            for (int j = 0; j < DC; ++j) s = s + a[j / 4][j % 4] * c[j / 4][j % 4];
        } else {
#pragma unroll
            for (int j = 0; j < DC; ++j)
                if (j < n) s = s + a[j / 4][j % 4] * c[j / 4][j % 4];
        }
    }
    return s;
}

// One lane per listed pair, grid-stride over the list's length on the device.
// SCORES: the score is qip's; otherwise the score rule's <u,q> is computed here
// and stored to qip for the top-k.
template <bool SCORES>
__global__ void __launch_bounds__(NT) k_list_exact(const float *__restrict__ users, const float *__restrict__ queries,
                                                   int32_t ld, int32_t dim, const float *__restrict__ table, int32_t S,
                                                   float eps, const float *__restrict__ gvals, FineCols fc,
                                                   const ListCounters *__restrict__ ctr, int64_t list_cap,
                                                   const int32_t *__restrict__ cl_u, const int32_t *__restrict__ cl_b,
                                                   int64_t n_user, uint32_t *__restrict__ bk_c,
                                                   float *__restrict__ qip, uint64_t *t) {
    stamp(t);
    __shared__ int32_t col[GW];
    __shared__ f32x4 sd[SCORES ? 1 : NT / 64][2][SCORES ? 1 : 64 * DP / 4];
    if (threadIdx.x < GW) col[threadIdx.x] = threadIdx.x < kMaxFine ? fc.col[threadIdx.x] : 0;
    __syncthreads();
    const int64_t n = list_len(ctr, list_cap);
    const int64_t per_round = (int64_t)gridDim.x * NT;
    for (int64_t r0 = 0; r0 < n; r0 += per_round) {
        const int64_t lb = xcd_block(min(n - r0, per_round));
        const int64_t w0 = r0 + lb * NT + (threadIdx.x & ~63);  // the wavefront's first pair
        if (lb < 0 || w0 >= n) continue;
        const int64_t i = r0 + lb * NT + threadIdx.x, ic = min(i, n - 1);
        const int64_t u = cl_u[ic], b = cl_b[ic];
        float s;
        if constexpr (SCORES) s = qip[b * n_user + u];
        else s = wave_rule_dot(sd[threadIdx.x >> 6][0], sd[threadIdx.x >> 6][1], users, queries, u, b, ld, dim);
        if (i >= n) continue;
        if (!SCORES) qip[b * n_user + u] = s;
        const float *row = table + u * (int64_t)S, *grow = gvals + u * GW;
        int32_t lo, hi;
        if (eps > 0.0f) {
            lo = bucket_of(grow, row, col, fc.n, S, __double2float_rd((double)s - (double)eps));
            hi = bucket_of(grow, row, col, fc.n, S, __double2float_ru((double)s + (double)eps));
        } else {
            lo = hi = bucket_of(grow, row, col, fc.n, S, s);
        }
        bk_c[i] = (uint32_t)lo | ((uint32_t)hi << 16);
    }
}

// Adds each lane's one (of the lanes that `on` says) to LDS bin j; lanes of the
// first two distinct bins add together, since many users of a popular query
// share a bucket.
__device__ __forceinline__ void add_bins(uint32_t *h, bool on, int32_t j) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const uint64_t todo = __builtin_amdgcn_ballot_w64(on);
        if (todo == 0) return;  // uniform
        const int l = __ffsll((unsigned long long)todo) - 1;
        const bool mine = on && j == __builtin_amdgcn_readlane(j, l);
        const uint64_t m = __builtin_amdgcn_ballot_w64(mine);
        if (lane == l) atomicAdd(&h[j], (uint32_t)__popcll(m));
        on = on && !mine;
    }
    if (on) atomicAdd(&h[j], 1u);
}

// Smallest bin j of h[0 .. FB) where `before` plus the counts up to j reach k:
// res = {j or -1, the sum up to j, the sum before j}; with j = -1 the sum is of
// all bins.  All threads call it.
constexpr int FB = 2048;
struct BinScan {
    int32_t bin;
    uint32_t upto, under;
};
template <int FT>
__device__ __forceinline__ void find_bin(const uint32_t *h, uint32_t before, uint32_t k, uint32_t *red, BinScan *res) {
    constexpr int PER = FB / FT;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    uint32_t v[PER], own = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        v[i] = h[threadIdx.x * PER + i];
        own += v[i];
    }
    uint32_t x = own;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) red[w] = x;
    __syncthreads();
    uint32_t sum = before, tot = before;
    for (int i = 0; i < FT / 64; ++i) {
        sum += i < w ? red[i] : 0u;
        tot += red[i];
    }
    sum += x - own;
    if (threadIdx.x == 0 && tot < k) *res = {-1, tot, tot};
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        if (sum < k && sum + v[i] >= k) *res = {(int32_t)threadIdx.x * PER + i, sum + v[i], sum};
        sum += v[i];
    }
    __syncthreads();
}

// One workgroup per query, over its pairs of the grouped list (FILTER: over the
// whole list of a few queries, skipping other queries' pairs): beta, the bucket
// of the k-th smallest b_lo, then the candidates (b_hi <= beta) with their rank
// when the bounds fix it, else ~(refine row).  A query with fewer than k buckets
// up to its threshold, or a list that overflowed, gets thr = -1 (the plan's own
// reasons stay) and no candidates: it is answered another way.
//
// Many candidates are users of bucket beta itself (an item that most of 100k
// users rank first).  When that bucket fixes the rank, the answer takes the
// smallest userIDs of it, as many as the buckets below leave: a histogram of
// their userIDs gives a bound, and the users past it are counted but not
// written, so the top-k sorts a few hundred keys and not 188k.
//
// Bound: latency of a few passes over some hundred pairs; a list of 250k pairs
// is read three times by one workgroup, 4096 pairs at a time.
template <bool FILTER, int FT>
__global__ void __launch_bounds__(FT) k_list_final(const int32_t *__restrict__ cl_u, const int32_t *__restrict__ cl_b,
                                                   const uint32_t *__restrict__ bk_c, const uint32_t *__restrict__ g_off,
                                                   const uint32_t *__restrict__ g_cnt, const float *__restrict__ qip,
                                                   ListCounters *__restrict__ ctr, int64_t list_cap, FineCols fc, int32_t S,
                                                   int same, const int32_t *__restrict__ ranks, int64_t n_item,
                                                   int64_t n_user, QueryInfo *__restrict__ qi,
                                                   int32_t *__restrict__ cand_user, int32_t *__restrict__ cand_rank,
                                                   int32_t *__restrict__ refine_user, int32_t *__restrict__ refine_query,
                                                   float *__restrict__ refine_thr, int32_t *__restrict__ cnt, uint64_t *t) {
    stamp(t);
    constexpr int UNR = 4096 / FT;
    __shared__ alignas(8) uint32_t h[FB];
    __shared__ uint32_t red[FT / 64];
    __shared__ BinScan s_beta, s_user;
    __shared__ int32_t s_cand, s_fill, s_refine;
    __shared__ int64_t s_off;
    const int32_t b = (int32_t)blockIdx.x;
    const int lane = threadIdx.x & 63;
    const QueryInfo q = qi[b];
    const bool listed = q.thr >= 0 && (int64_t)ctr->n_list <= list_cap;  // list_len, and thr = -1 past it
    const int64_t first = !listed || FILTER ? 0 : g_off[b];
    const int64_t end = !listed ? 0 : FILTER ? (int64_t)ctr->n_list : first + g_cnt[b];
    const uint32_t k = (uint32_t)q.topk;
    if (threadIdx.x == 0) { s_beta = {-1, 0u, 0u}; s_cand = s_fill = s_refine = 0; }
    // buckets of UNR pairs per thread, loads in flight together; bit 31 of none: not a pair of b
    constexpr uint32_t none = 0xFFFFFFFFu;
    auto load = [&](int64_t i0, uint32_t (&x)[UNR]) {
        int32_t y[UNR];
#pragma unroll
        for (int j = 0; j < UNR; ++j) {  // the last pair again past the end: no branch between the loads
            const int64_t i = min(i0 + j * FT + threadIdx.x, end - 1);
            x[j] = bk_c[i];
            y[j] = FILTER ? cl_b[i] : b;
        }
#pragma unroll
        for (int j = 0; j < UNR; ++j)
            if (i0 + j * FT + threadIdx.x >= end || y[j] != b) x[j] = none;
    };
    // beta: only buckets up to the threshold can hold it
    const int32_t last = listed ? fc.col[q.thr] : -1;
    uint32_t before = 0;
    int32_t beta = -1;
    __syncthreads();
    for (int32_t w0 = 0; w0 <= last && beta < 0; w0 += FB) {
        for (int j = threadIdx.x; j < FB; j += FT) h[j] = 0u;
        __syncthreads();
        for (int64_t i0 = first; i0 < end; i0 += FT * UNR) {
            uint32_t x[UNR];
            load(i0, x);
#pragma unroll
            for (int j = 0; j < UNR; ++j) {
                const int32_t lo = (int32_t)(x[j] & 0xFFFFu);
                add_bins(h, x[j] != none && lo >= w0 && lo <= min(last, w0 + FB - 1), lo - w0);
            }
        }
        __syncthreads();
        find_bin<FT>(h, before, k, red, &s_beta);
        before = s_beta.upto;
        if (s_beta.bin >= 0) beta = w0 + s_beta.bin;
        __syncthreads();  // s_beta is read before the next window's
    }
    if (beta < 0) {  // uniform
        if (threadIdx.x == 0) {
            qi[b].beta = qi[b].gamma = -1;
            if (q.thr >= 0) qi[b].thr = -1;
            qi[b].n_cand = qi[b].n_dropped = qi[b].n_refine = qi[b].fill = qi[b].n_settled = 0;
            qi[b].cand_off = 0;
        }
        return;
    }
    const uint32_t under = s_beta.under;  // pairs with b_lo < beta
    uint32_t n_cand = s_beta.upto;
    if (!same) {
        int32_t c = 0;
        for (int64_t i0 = first; i0 < end; i0 += FT * UNR) {
            uint32_t x[UNR];
            load(i0, x);
#pragma unroll
            for (int j = 0; j < UNR; ++j) c += x[j] != none && (int32_t)(x[j] >> 16) <= beta;
        }
        if (c) atomicAdd(&s_cand, c);
        __syncthreads();
        n_cand = (uint32_t)s_cand;
    }
    auto rank_lb = [&](int32_t j) { return j == S ? (int32_t)n_item : ranks[j]; };
    auto rank_ub = [&](int32_t j) { return j == 0 ? 0 : ranks[j - 1] + 1; };
    // the users of bucket beta that the answer can hold
    int32_t u_max = INT32_MAX;
    uint32_t n_keep = n_cand;
    if (same && n_cand > 1024u && rank_lb(beta) == rank_ub(beta)) {  // uniform
        int sh = 0;
        while (((n_user - 1) >> sh) >= FB) ++sh;
        for (int j = threadIdx.x; j < FB; j += FT) h[j] = 0u;
        __syncthreads();
        for (int64_t i0 = first; i0 < end; i0 += FT * UNR) {
            uint32_t x[UNR];
            load(i0, x);
            int32_t u[UNR];
#pragma unroll
            for (int j = 0; j < UNR; ++j) u[j] = cl_u[min(i0 + j * FT + threadIdx.x, end - 1)];
#pragma unroll
            for (int j = 0; j < UNR; ++j)
                if (x[j] != none && (int32_t)(x[j] >> 16) == beta) atomicAdd(&h[u[j] >> sh], 1u);
        }
        __syncthreads();
        find_bin<FT>(h, under, k, red, &s_user);  // found: bucket beta reaches k
        u_max = (int32_t)(((int64_t)s_user.bin + 1) << sh) - 1;
        n_keep = s_user.upto;
    }
    if (threadIdx.x == 0) s_off = atomicAdd(&ctr->n_cand, (int32_t)n_keep);
    __syncthreads();
    const int64_t off = s_off;
    // refine rows (user, candidate slot) until their number is known, in the histogram's place
    constexpr int ROWS = FB / 2;
    uint2 *rows = reinterpret_cast<uint2 *>(h);
    auto refine_row = [&](int32_t r, int32_t u) {
        refine_user[r] = u;
        refine_query[r] = b;
        refine_thr[r] = qip[(int64_t)b * n_user + u];
        cnt[r] = 0;
    };
    for (int64_t i0 = first; i0 < end; i0 += FT * UNR) {
        uint32_t x[UNR];
        int32_t us[UNR];
        load(i0, x);
#pragma unroll
        for (int j = 0; j < UNR; ++j) us[j] = cl_u[min(i0 + j * FT + threadIdx.x, end - 1)];
#pragma unroll
        for (int j = 0; j < UNR; ++j) {
            const int32_t u = us[j];
            const int32_t blo = (int32_t)(x[j] & 0xFFFFu), bhi = (int32_t)(x[j] >> 16);
            const bool cand = x[j] != none && (bhi < beta || (bhi == beta && u <= u_max));
            const uint64_t m = __builtin_amdgcn_ballot_w64(cand);
            if (m == 0) continue;  // uniform in the wavefront
            int32_t rank = 0;
            bool open = false;
            if (cand) {
                rank = rank_lb(blo);
                open = rank != rank_ub(bhi);
            }
            int32_t place = 0;
            if (lane == 0) place = atomicAdd(&s_fill, (int32_t)__popcll(m));
            place = __shfl(place, 0, 64) + (int32_t)__popcll(m & ((1ull << lane) - 1));
            if (open) {
                const int32_t r = atomicAdd(&s_refine, 1);
                if (r < ROWS) {
                    rows[r] = make_uint2((uint32_t)u, (uint32_t)place);
                } else {
                    const int32_t g = atomicAdd(&ctr->n_refine, 1);
                    refine_row(g, u);
                    rank = ~g;
                }
            }
            if (cand) {
                cand_user[off + place] = u;
                cand_rank[off + place] = rank;
            }
        }
    }
    __syncthreads();
    const int32_t n_rows = min(s_refine, ROWS);
    if (threadIdx.x == 0 && n_rows > 0) s_cand = atomicAdd(&ctr->n_refine, n_rows);
    __syncthreads();
    for (int32_t i = threadIdx.x; i < n_rows; i += FT) {
        const int32_t r = s_cand + i;
        refine_row(r, (int32_t)rows[i].x);
        cand_rank[off + rows[i].y] = ~r;
    }
    if (threadIdx.x == 0) {
        QueryInfo r = q;
        r.beta = r.gamma = beta;
        r.n_cand = (int32_t)n_cand;
        r.n_dropped = (int32_t)(n_cand - n_keep);
        r.n_refine = s_refine;
        r.fill = (int32_t)n_keep;
        r.n_settled = 0;
        r.cand_off = off;
        qi[b] = r;
    }
}

// gv[u * kGuardRow + f] = gc[f * pitch + u] = T[u][col_f], -inf past the fine
// columns, rows [u0, u0 + n_rows): by rows for the searches of one user, by
// columns (if gc) for the lists, which read one column of many users.
__global__ void __launch_bounds__(NT) k_gather_guards(const float *__restrict__ T, int64_t S, FineCols fc, int64_t u0,
                                                      int64_t n_rows, float *__restrict__ gv, float *__restrict__ gc,
                                                      int64_t pitch) {
    __shared__ float tile[64][GP];
    const int64_t r0 = (int64_t)blockIdx.x * 64;
#pragma unroll 4
    for (int i = threadIdx.x; i < 64 * GW; i += NT) {
        const int r = i / GW, f = i % GW;
        if (r0 + r >= n_rows) break;
        const int64_t u = u0 + r0 + r;
        const float v = f < fc.n ? T[u * S + fc.col[f]] : -INFINITY;
        gv[u * GW + f] = v;
        tile[r][f] = v;
    }
    if (!gc) return;
    __syncthreads();
    for (int i = threadIdx.x; i < 64 * GW; i += NT) {
        const int f = i / 64, r = i % 64;
        if (r0 + r < n_rows) gc[f * pitch + u0 + r0 + r] = tile[r][f];
    }
}

// Moves rows rows[0] < rows[1] < ... of x to rows 0, 1, ...: a thread per
// column, eight rows read before any of their places is written (a later row's
// source lies behind them, rows[i] >= i).
__global__ void __launch_bounds__(NT) k_keep_rows(float *__restrict__ x, int64_t n_col, const int32_t *__restrict__ rows, int32_t n) {
    const int64_t u = (int64_t)blockIdx.x * NT + threadIdx.x;
    if (u >= n_col) return;
    for (int32_t i = 0; i < n; i += 8) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = x[(int64_t)rows[min(i + j, n - 1)] * n_col + u];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (i + j < n) x[(int64_t)(i + j) * n_col + u] = v[j];
    }
}

bool fine_ok(const FineCols &fc, int64_t S) {
    if (fc.n < 1 || fc.n > kMaxFine) return false;
    for (int f = 0; f < fc.n; ++f)
        if (fc.col[f] < 0 || fc.col[f] >= S || (f > 0 && fc.col[f] <= fc.col[f - 1])) return false;
    return true;
}

}  // namespace

hipError_t launch_gather_guards(hipStream_t s, const float *T, int64_t S, const FineCols &fc, int64_t u0,
                                int64_t n_rows, float *gv, float *gc, int64_t pitch) {
    if (n_rows <= 0) return hipSuccess;
    if ((fc.n > 0 && !fine_ok(fc, S)) || u0 + n_rows > pitch) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_gather_guards, dim3((unsigned)((n_rows + 63) / 64)), dim3(NT), 0, s, T, S, fc, u0, n_rows, gv,
                       gc, pitch);
    return hipGetLastError();
}

hipError_t launch_keep_rows(hipStream_t s, float *x, int64_t n_col, const int32_t *rows, int32_t n) {
    if (n <= 0 || n_col <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_keep_rows, dim3((unsigned)((n_col + NT - 1) / NT)), dim3(NT), 0, s, x, n_col, rows, n);
    return hipGetLastError();
}

#define RKR_KS_SWITCH(kp, CASE)             \
    switch ((kp) / 32) {                    \
        CASE(1) CASE(2) CASE(3) CASE(4)     \
        CASE(5) CASE(6) CASE(7) CASE(8)     \
        default: return hipErrorInvalidValue; \
    }

hipError_t launch_list_screen(hipStream_t s, const ListLaunch &L) {
    if (L.nq <= 0 || L.n_user <= 0) return hipSuccess;
    if (!fine_ok(L.fc, L.S) || !L.gvals || !L.gcols || L.pitch < L.n_user || !L.user_hi || !L.q_hi) return hipErrorInvalidValue;
    if (L.products != 1 && (L.products != 3 || !L.user_lo || !L.q_lo)) return hipErrorInvalidValue;
    ListScreen P{L.user_hi, L.user_lo, L.user_norm, L.gvals, L.gcols, L.pitch, L.q_hi, L.q_lo, L.q_cs, L.nq, L.Kp, L.fc.n,
                 L.C, L.floor};
    const int64_t n_s = (L.n_user + L.stride - 1) / L.stride, n_sb = (n_s + 127) / 128;
    const unsigned qg = (unsigned)((L.nq + QST - 1) / QST);
    // two workgroups of the sample fit a CU
    const unsigned gx = (unsigned)std::max<int64_t>(1, std::min<int64_t>(n_sb, (2 * L.n_cu + qg - 1) / qg));
#define RKR_SAMPLE_CASE(ks)                                                                                       \
    case ks:                                                                                                      \
        if (L.products == 1)                                                                                      \
            hipLaunchKernelGGL((k_sample_screen<ks, 1>), dim3(gx, qg), dim3(NT), 0, s, P, n_s, L.stride, L.n_user, L.hist); \
        else                                                                                                      \
            hipLaunchKernelGGL((k_sample_screen<ks, 3>), dim3(gx, qg), dim3(NT), 0, s, P, n_s, L.stride, L.n_user, L.hist); \
        break;
    RKR_KS_SWITCH(L.Kp, RKR_SAMPLE_CASE)
#undef RKR_SAMPLE_CASE
    hipLaunchKernelGGL(k_list_plan, dim3(1), dim3(PT), 0, s, L.hist, L.nq, L.fc.n, L.stride, L.n_user, L.cap, L.share,
                       L.band, L.room, L.list_cap, L.fc.coarse, L.qi, L.order, L.colg, L.ctr);
    // users per unit and workgroups per CU
    const bool wide = L.products == 1 && L.Kp <= 160;
    const int64_t ub = wide ? 256 : 128;
    const int64_t units = (L.n_user + ub - 1) / ub * ((L.nq + kSlice - 1) / kSlice);
    const dim3 grid((unsigned)std::max<int64_t>(1, std::min<int64_t>(units, (int64_t)L.n_cu * (wide ? 3 : 2))));
#define RKR_LIST_CASE(ks)                                                                                          \
    case ks:                                                                                                       \
        if (L.products == 1)                                                                                       \
            hipLaunchKernelGGL((k_list_screen<ks, ks <= 5 ? 4 : 2, 1>), grid, dim3(NT), 0, s, P, L.n_user, L.order, \
                               L.colg, L.g_cnt, L.ctr, L.raw_u, L.raw_b, L.list_cap);                              \
        else                                                                                                       \
            hipLaunchKernelGGL((k_list_screen<ks, 2, 3>), grid, dim3(NT), 0, s, P, L.n_user, L.order, L.colg,      \
                               L.g_cnt, L.ctr, L.raw_u, L.raw_b, L.list_cap);                                      \
        break;
    RKR_KS_SWITCH(L.Kp, RKR_LIST_CASE)
#undef RKR_LIST_CASE
    return hipGetLastError();
}

hipError_t launch_list_scores(hipStream_t s, const ListLaunch &L) {
    if (L.nq <= 0 || L.n_user <= 0) return hipSuccess;
    if (!fine_ok(L.fc, L.S) || !L.gvals || !L.gcols || L.pitch < L.n_user) return hipErrorInvalidValue;
    const int64_t n_s = (L.n_user + L.stride - 1) / L.stride;
    const unsigned qg = (unsigned)((L.nq + 15) / 16);
    const unsigned gx = (unsigned)std::max<int64_t>(1, std::min<int64_t>((n_s + 63) / 64, (8 * L.n_cu + qg - 1) / qg));
    hipLaunchKernelGGL(k_sample_scores, dim3(gx, qg), dim3(NT), 0, s, L.qip, L.n_user, L.nq, L.eps, L.gvals, L.fc.n,
                       n_s, L.stride, L.hist, L.t_bound);
    hipLaunchKernelGGL(k_list_plan, dim3(1), dim3(PT), 0, s, L.hist, L.nq, L.fc.n, L.stride, L.n_user, L.cap, L.share,
                       L.band, L.room, L.list_cap, L.fc.coarse, L.qi, L.order, L.colg, L.ctr);
    hipLaunchKernelGGL(k_list_scores,
                       dim3((unsigned)((L.n_user + NT - 1) / NT), (unsigned)((L.nq + kScoreSlice - 1) / kScoreSlice)),
                       dim3(NT), 0, s, L.qip, L.n_user, L.eps, L.gcols, L.pitch, L.order, L.colg, L.nq, L.g_cnt, L.ctr,
                       L.raw_u, L.raw_b, L.list_cap);
    return hipGetLastError();
}

hipError_t launch_list_exact(hipStream_t s, const ListLaunch &L, const float *users, const float *queries, int32_t ld,
                             int32_t dim, const float *table, bool scores, uint32_t *bk_c) {
    if (L.nq <= 0 || L.n_user <= 0) return hipSuccess;
    uint64_t *t = scores ? nullptr : L.t_bound;
    if (L.g_cnt) {
        const dim3 cg((unsigned)std::max(1, L.n_cu / 2));
        hipLaunchKernelGGL(k_list_count, cg, dim3(CT), 0, s, L.raw_b, L.list_cap, L.nq, L.g_cnt, L.ctr, t);
        hipLaunchKernelGGL(k_list_scatter, cg, dim3(CT), 0, s, L.raw_u, L.raw_b, L.list_cap, L.nq, L.g_cnt, L.g_off,
                           L.g_cur, L.ctr, L.cl_u, L.cl_b);
        t = nullptr;
    }
    const dim3 grid((unsigned)(L.n_cu * 16));  // a multiple of the 8 XCDs (grid-stride over the list)
    if (scores)
        hipLaunchKernelGGL(k_list_exact<true>, grid, dim3(NT), 0, s, users, queries, ld, dim, table, L.S, L.eps, L.gvals,
                           L.fc, L.ctr, L.list_cap, L.cl_u, L.cl_b, L.n_user, bk_c, L.qip, t);
    else
        hipLaunchKernelGGL(k_list_exact<false>, grid, dim3(NT), 0, s, users, queries, ld, dim, table, L.S, L.eps, L.gvals,
                           L.fc, L.ctr, L.list_cap, L.cl_u, L.cl_b, L.n_user, bk_c, L.qip, t);
    return hipGetLastError();
}

hipError_t launch_list_final(hipStream_t s, const ListLaunch &L, const uint32_t *bk_c, const int32_t *ranks,
                             int64_t n_item, int32_t *cand_user, int32_t *cand_rank, int32_t *refine_user,
                             int32_t *refine_query, float *refine_thr, int32_t *cnt) {
    if (L.nq <= 0 || L.n_user <= 0) return hipSuccess;
    const dim3 grid((unsigned)L.nq);
    const int same = L.eps > 0.0f ? 0 : 1;
    if (L.g_cnt)
        hipLaunchKernelGGL((k_list_final<false, 512>), grid, dim3(512), 0, s, L.cl_u, L.cl_b, bk_c, L.g_off, L.g_cnt, L.qip, L.ctr,
                           L.list_cap, L.fc, L.S, same, ranks, n_item, L.n_user, L.qi, cand_user, cand_rank, refine_user,
                           refine_query, refine_thr, cnt, L.t_prune);
    else
        hipLaunchKernelGGL((k_list_final<true, 1024>), grid, dim3(1024), 0, s, L.cl_u, L.cl_b, bk_c, nullptr, nullptr, L.qip, L.ctr,
                           L.list_cap, L.fc, L.S, same, ranks, n_item, L.n_user, L.qi, cand_user, cand_rank, refine_user,
                           refine_query, refine_thr, cnt, L.t_prune);
    return hipGetLastError();
}

}  // namespace rkr
