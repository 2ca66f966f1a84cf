// rkr_api.cpp -- the C ABI of librkr.so (include/rkr.h): context, resident
// device data, table build and the batched query pipeline.  Host-side logic
// only; every score, bound, count and selection runs in the HIP kernels.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <string>
#include <string_view>
#include <unordered_map>
#include <thread>
#include <vector>

#include "rkr_internal.hpp"

namespace rkr {

int set_err(Ctx *c, int code, const std::string &msg) {
    if (c) {
        std::lock_guard<std::mutex> g(c->err_mu);
        c->err = msg;
    }
    return code;
}

const char *kVersion = "rkr 0.1 (gfx950)";

// Frees the build scratch if no call is using it (mem_mu is held).
static bool drop_misc(Ctx *c) {
    if (c->misc_busy || !c->misc.p) return false;
    const auto it = c->alloc_bytes.find(c->misc.p);
    (void)hipFree(c->misc.p);
    c->held -= std::min(c->held, it->second);
    c->alloc_bytes.erase(it);
    c->misc = DeviceBuf{};
    return true;
}

size_t free_bytes(Ctx *c) {
    std::lock_guard<std::mutex> g(c->mem_mu);
    return (c->budget > c->held ? c->budget - c->held : 0) + (c->misc_busy ? 0 : c->misc.bytes);
}

int dev_alloc(Ctx *c, void **p, size_t bytes, const char *what) {
    *p = nullptr;
    if (bytes == 0) return RKR_OK;
    std::lock_guard<std::mutex> g(c->mem_mu);
    if (c->held + bytes > c->budget) (void)drop_misc(c);
    if (c->held + bytes > c->budget)
        return set_err(c, RKR_ERR_NOMEM, std::string("device memory budget exceeded allocating ") + what + " (" +
                                             std::to_string(bytes) + " bytes, budget " + std::to_string(c->budget) +
                                             ", held " + std::to_string(c->held) + ")");
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess && drop_misc(c)) {
        (void)hipGetLastError();
        e = hipMalloc(p, bytes);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        *p = nullptr;
        return set_err(c, RKR_ERR_NOMEM, std::string("hipMalloc ") + what + ": " + hipGetErrorString(e));
    }
    c->held += bytes;
    c->alloc_bytes[*p] = bytes;
    return RKR_OK;
}

namespace {
thread_local bool tl_defer_frees = false;
}

void set_defer_frees(bool on) { tl_defer_frees = on; }
bool defer_frees() { return tl_defer_frees; }

// The size recorded at allocation is what returns to the budget; `bytes` is
// only used for a pointer this context did not allocate.
void dev_free(Ctx *c, void *p, size_t bytes) {
    if (!p) return;
    std::lock_guard<std::mutex> g(c->mem_mu);
    auto it = c->alloc_bytes.find(p);
    if (it != c->alloc_bytes.end()) {
        bytes = it->second;
        c->alloc_bytes.erase(it);
    }
    if (tl_defer_frees) {
        c->retired.push_back({p, bytes});
        return;
    }
    (void)hipFree(p);
    c->held -= std::min(c->held, bytes);
}

void release_retired(Ctx *c) {
    std::lock_guard<std::mutex> g(c->mem_mu);
    for (const auto &r : c->retired) {
        (void)hipFree(r.p);
        c->held -= std::min(c->held, r.bytes);
    }
    c->retired.clear();
}

DataSnap snap_of(const Ctx *c) {
    DataSnap d;
    d.n_user = c->n_user;
    d.n_item = c->n_item;
    d.n_item_base = c->n_item_base;
    d.users = c->users;
    d.usersT = c->usersT;
    d.items = c->items;
    d.user_norm = c->user_norm;
    d.rho = c->rho;
    d.user_hi = c->user_hi;
    d.user_lo = c->user_lo;
    d.item_norm = c->item_norm;
    d.item_hi = c->item_hi;
    d.item_lo = c->item_lo;
    d.table = c->table;
    d.side_ins = c->side_ins;
    d.side_del = c->side_del;
    d.n_ins = c->n_ins;
    d.n_del = c->n_del;
    d.ld_ins = c->ld_ins;
    d.ld_del = c->ld_del;
    d.max_abs_user = c->max_abs_user;
    d.screen_abs = c->screen_abs;
    d.qtable = c->qtable;
    d.qranks = c->qranks;
    d.n_qs = c->n_qs;
    d.fine = c->fine;
    d.guards = c->guards;
    d.gvals = c->gvals;
    d.gcols = c->gcols;
    d.gpitch = c->gpitch;
    d.ranks = c->ranks;
    d.n_sample = c->n_sample;
    d.table_eps = c->table_eps;
    d.qcol = c->qcol;
    d.hrk = c->hrk;
    for (int j = 0; j < 8; ++j) d.ins_gmax[j] = c->ins_gmax[j];
    if (c->qsrp_users && c->qsrp_n_user == c->n_user) {
        d.qsrp_users = c->qsrp_users;
        d.qsrp_rot = c->qsrp_rot;
        d.qsrp_par = c->qsrp_par;
        d.qsrp_cd = c->qsrp_cd;
        d.qsrp_ldr = c->qsrp_ldr;
        d.qsrp_gcd = c->qsrp_gcd;
        d.qsrp_crot = c->qsrp_crot;
    }
    return d;
}

// 64-bit hash of n bytes salted with `salt`: four independent multiply-add
// lanes over 8-byte words (zero-padded tail), then an xorshift-multiply fold.
// The dedup key of a query row; equal hashes are confirmed by a byte compare.
uint64_t row_hash(const void *p, size_t n, uint32_t salt) {
    const unsigned char *b = static_cast<const unsigned char *>(p);
    const uint64_t m = 0xBF58476D1CE4E5B9ull;
    uint64_t h[4] = {0x9E3779B97F4A7C15ull ^ n, 0xC2B2AE3D27D4EB4Full ^ salt, 0x165667B19E3779F9ull,
                     0xD6E8FEB86659FD93ull};
    size_t i = 0;
    for (; i + 32 <= n; i += 32) {
        uint64_t w[4];
        std::memcpy(w, b + i, 32);
        for (int l = 0; l < 4; ++l) h[l] = (h[l] + w[l]) * m;
    }
    if (i < n) {
        uint64_t w[4] = {0, 0, 0, 0};
        std::memcpy(w, b + i, n - i);
        for (int l = 0; l < 4; ++l) h[l] = (h[l] + w[l]) * m;
    }
    uint64_t x = (h[0] ^ (h[0] >> 29)) + 3 * (h[1] ^ (h[1] >> 31)) + 5 * (h[2] ^ (h[2] >> 27)) +
                 7 * (h[3] ^ (h[3] >> 33));
    x ^= x >> 29;
    x *= 0x94D049BB133111EBull;
    return x ^ (x >> 32);
}

namespace {
// The table columns nearest below ranks 4^j - 1 (3, 15, ..., 16383), at most
// 7, ascending.
int guard_table_columns(const std::vector<int32_t> &hr, int32_t *col) {
    int n = 0;
    int32_t last = -1;
    for (int64_t target = 3; target <= 16383 && n < 7; target = target * 4 + 3) {
        const auto it = std::upper_bound(hr.begin(), hr.end(), (int32_t)target);
        const int32_t j = (int32_t)(it - hr.begin()) - 1;
        if (j > last) {
            col[n++] = j;
            last = j;
        }
    }
    return n;
}
}  // namespace

// The guard columns and, inside each of their bins and past the last one, up
// to 7 more spaced geometrically in rank: neighbouring fine columns differ by a
// factor of about 1.2 in rank (4 between guard columns), which is how much a
// list is longer than it has to be.
static FineCols fine_columns(const std::vector<int32_t> &hr) {
    FineCols fc{};
    if (hr.empty()) return fc;
    int32_t gcol[8];
    const int ng = guard_table_columns(hr, gcol);
    int32_t last = -1;
    auto take = [&](int32_t j, bool coarse) {
        if (j <= last || fc.n >= kMaxFine) return;
        if (coarse) fc.coarse |= 1ull << fc.n;
        fc.col[fc.n++] = j;
        last = j;
    };
    for (int g = 0; g <= ng; ++g) {
        const int32_t lo = last + 1, hi = g < ng ? gcol[g] : (int32_t)hr.size() - 1;
        if (lo > hi) continue;
        const double ra = (double)hr[lo] + 1.0, rb = (double)hr[hi] + 1.0;
        for (int m = 0; m < 7; ++m) {
            const auto it = std::upper_bound(hr.begin() + lo, hr.begin() + hi, (int32_t)(ra * std::pow(rb / ra, m / 7.0) - 1.0));
            const int32_t j = (int32_t)(it - hr.begin()) - 1;
            if (j >= lo && j < hi) take(j, false);
        }
        take(hi, g < ng);
    }
    return fc;
}

void set_table_columns(Ctx *c) {
    c->hrk = std::make_shared<const std::vector<int32_t>>(c->qtable ? c->h_qranks : c->h_ranks);
    c->fine = fine_columns(*c->hrk);
    c->guards = GuardCols{};
    for (int f = 0; f < c->fine.n; ++f)
        if ((c->fine.coarse >> f) & 1) {
            c->guards.col[c->guards.n] = c->fine.col[f];
            c->guards.idx[c->guards.n++] = f;
        }
}

int refresh_guard_values(Ctx *c, int64_t u0, int64_t n) {
    if (!c->gvals || n <= 0) return RKR_OK;
    const float *T = c->qtable ? c->qtable : c->table;
    const int64_t S = c->qtable ? c->n_qs : c->n_sample;
    RKR_HIP(c, launch_gather_guards(c->stream, T, S, c->fine, u0, n, c->gvals, c->gcols, c->gpitch));
    return RKR_OK;
}

// Guard rows and columns, one allocation.  The columns only spare the lists a
// stride of 64 floats; where they would take what a query needs there are rows
// only, and queries are searched.
static size_t guard_bytes(int64_t cap, bool cols) { return sizeof(float) * (cols ? 2 : 1) * (size_t)cap * kGuardRow; }

int new_guards(Ctx *c, int64_t cap, size_t spare, Guards *g) {
    g->cap = cap;
    g->cols = free_bytes(c) >= 3 * guard_bytes(cap, false) + spare;
    return dev_alloc_t(c, &g->p, guard_bytes(cap, g->cols) / sizeof(float), "guard values");
}

void place_guards(Ctx *c, const Guards &g) {
    if (g.p != c->gvals) dev_free(c, c->gvals, 0);
    c->gvals = g.p;
    c->gcols = g.cols ? g.p + (size_t)g.cap * kGuardRow : nullptr;
    c->gpitch = g.cap;
}

int alloc_guards(Ctx *c, int64_t cap, size_t spare) {
    Guards g;
    if (int rc = new_guards(c, cap, spare, &g)) return rc;
    place_guards(c, g);
    return RKR_OK;
}

// p if it is an allocation of `bytes` that no batch can be reading (p is then
// null: the buffer is the caller's), else null.
template <class T>
static T *keep_buffer(Ctx *c, T *&p, size_t bytes) {
    if (!p || bytes == 0 || defer_frees()) return nullptr;
    std::lock_guard<std::mutex> g(c->mem_mu);
    const auto it = c->alloc_bytes.find(p);
    if (it == c->alloc_bytes.end() || it->second != bytes) return nullptr;
    T *const q = p;
    p = nullptr;
    return q;
}

std::vector<int32_t> query_table_ranks(const std::vector<int32_t> &sample, int64_t n_item, int mode) {
    std::vector<int32_t> r(sample);
    if (mode == 2) {
        // every rank below D, with D as large as the column cap allows
        int64_t lo = 0, hi = std::min<int64_t>(n_item, kMaxSample);
        while (lo < hi) {
            const int64_t D = (lo + hi + 1) / 2;
            int64_t above = 0;
            for (int32_t x : sample) above += x >= D ? 1 : 0;
            if (D + above <= kMaxSample) lo = D; else hi = D - 1;
        }
        for (int64_t x = 0; x < lo; ++x) r.push_back((int32_t)x);
    } else {
        for (int64_t x = 0; x < 256; ++x) r.push_back((int32_t)x);
        for (int64_t x = 256; x < 1024; x += 8) r.push_back((int32_t)x);
        for (int64_t x = 1024; x < 4096; x += 32) r.push_back((int32_t)x);
    }
    std::vector<int32_t> out;
    std::sort(r.begin(), r.end());
    for (int32_t x : r)
        if (x < n_item && (out.empty() || x != out.back())) out.push_back(x);
    if ((int64_t)out.size() > kMaxSample) out.clear();
    return out;
}

// Grow-only scratch buffer.
int ensure(Ctx *c, DeviceBuf &b, size_t bytes, const char *what) {
    if (b.bytes >= bytes) return RKR_OK;
    dev_free(c, b.p, b.bytes);
    b.p = nullptr;
    b.bytes = 0;
    size_t want = std::max(bytes, b.bytes * 3 / 2);
    int rc = dev_alloc(c, &b.p, want, what);
    if (rc != RKR_OK) {
        rc = dev_alloc(c, &b.p, bytes, what);
        if (rc != RKR_OK) return rc;
        want = bytes;
    }
    b.bytes = want;
    return RKR_OK;
}

int ensure_pinned(Ctx *c, PinnedBuf &b, size_t bytes) {
    if (b.bytes >= bytes) return RKR_OK;
    free_pinned(b);
    const size_t want = std::max(bytes, b.bytes + b.bytes / 2);
    // coherent: kernels read and write it beside the host
    if (hipHostMalloc(&b.p, want, hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess) {
        b.p = nullptr;
        return set_err(c, RKR_ERR_NOMEM, "pinned host staging (" + std::to_string(want) + " bytes)");
    }
    b.bytes = want;
    return RKR_OK;
}

void free_pinned(PinnedBuf &b) {
    if (b.p) (void)hipHostFree(b.p);
    b.p = nullptr;
    b.bytes = 0;
}

void free_qsrp(Ctx *c) {
    for (float *p : {c->qsrp_users, c->qsrp_rot, c->qsrp_par}) dev_free(c, p, 0);
    c->qsrp_users = c->qsrp_rot = c->qsrp_par = nullptr;
    c->qsrp_cd = c->qsrp_ldr = 0;
    c->qsrp_n_user = c->qsrp_fallback = 0;
}

namespace {

// Forgets the pending item updates.  keep_buffers leaves the side arrays and
// item lists allocated at their row lengths and capacities for the inserts
// that follow a rebuild (a serving loop's memory stays flat); with two buffers
// per side the next update writes the one no batch of the new state reads.
void free_update_state(Ctx *c, bool keep_buffers = false) {
    if (!keep_buffers) {
        for (float *p : {c->items_ins, c->items_del, c->side_ins, c->side_del, c->side_ins_spare, c->side_del_spare})
            dev_free(c, p, 0);
        c->items_ins = c->items_del = c->side_ins = c->side_del = nullptr;
        c->side_ins_spare = c->side_del_spare = nullptr;
        c->ld_ins = c->ld_del = 0;
        c->ins_cap = c->del_cap = 0;
    }
    c->n_ins = c->n_del = 0;
    for (int j = 0; j < 8; ++j) c->ins_gmax[j] = 0;
    if (c->items_base && c->items_base != c->items)
        dev_free(c, c->items_base, sizeof(float) * (size_t)c->n_item_base * c->ld);
    c->items_base = c->items;
    c->n_item_base = c->n_item;
    c->cur_src.clear();
    c->base_deleted.clear();
}

void free_table(Ctx *c) {
    free_qsrp(c);  // fitted to this table
    dev_free(c, c->ranks, 0);
    dev_free(c, c->table, 0);
    dev_free(c, c->qranks, 0);
    dev_free(c, c->qcol, 0);
    dev_free(c, c->qtable, 0);
    dev_free(c, c->gvals, 0);
    c->gcols = nullptr;
    c->gpitch = 0;
    c->ranks = c->qranks = c->qcol = nullptr;
    c->table = c->qtable = c->gvals = nullptr;
    c->n_sample = c->n_qs = 0;
    c->h_ranks.clear();
    c->h_qranks.clear();
    set_table_columns(c);
    c->table_eps = 0.0f;
}

void free_data(Ctx *c) {
    free_update_state(c);
    free_table(c);
    dev_free(c, c->upd_scratch.p, 0);
    c->upd_scratch = DeviceBuf{};
    c->u_cap = c->i_cap = 0;
    const size_t ld = (size_t)c->ld;
    dev_free(c, c->users, sizeof(float) * (size_t)c->n_user * ld);
    dev_free(c, c->usersT, sizeof(float) * (size_t)((c->n_user + 63) / 64) * 64 * ld);
    dev_free(c, c->items, sizeof(float) * (size_t)c->n_item * ld);
    dev_free(c, c->item_hi, sizeof(uint16_t) * (size_t)c->n_item * c->kp);
    dev_free(c, c->item_lo, sizeof(uint16_t) * (size_t)c->n_item * c->kp);
    dev_free(c, c->item_norm, sizeof(float) * (size_t)c->n_item);
    dev_free(c, c->user_norm, sizeof(float) * (size_t)c->n_user);
    dev_free(c, c->user_hi, 0);
    dev_free(c, c->user_lo, 0);
    c->user_hi = c->user_lo = nullptr;
    c->item_hi = c->item_lo = nullptr;
    c->item_norm = c->user_norm = nullptr;
    c->kp = 0;
    c->users = c->usersT = c->items = nullptr;
    c->items_base = nullptr;  // it was c->items by now
    c->n_user = c->n_item = 0;
    c->dim = c->ld = 0;
}

void free_bufs(Ctx *c, std::initializer_list<DeviceBuf *> bufs) {
    for (DeviceBuf *b : bufs) {
        dev_free(c, b->p, b->bytes);
        b->p = nullptr;
        b->bytes = 0;
    }
}

void free_scratch(Ctx *c) {
    Slot &s = c->main;
    free_bufs(c, {&s.io, &s.qip, &s.bk, &s.cand, &s.refine_idx, &s.recheck, &s.hist, &s.q_split, &s.list_info, &s.list, &c->misc});
}

}  // namespace

int slot_init(Ctx *c, Slot &sl, bool own_stream, const std::vector<uint32_t> *cu_mask) {
    sl.own_stream = own_stream;
    if (own_stream && cu_mask) {
        RKR_HIP(c, hipExtStreamCreateWithCUMask(&sl.stream, (uint32_t)cu_mask->size(), cu_mask->data()));
    } else if (own_stream) {
        RKR_HIP(c, hipStreamCreateWithFlags(&sl.stream, hipStreamNonBlocking));
    } else {
        sl.stream = c->stream;
    }
    for (auto &e : sl.ev) RKR_HIP(c, hipEventCreate(&e));
    return RKR_OK;
}

void slot_free(Ctx *c, Slot &sl) {
    if (sl.stream) (void)hipStreamSynchronize(sl.stream);
    free_bufs(c, {&sl.io, &sl.qip, &sl.bk, &sl.cand, &sl.refine_idx, &sl.recheck, &sl.hist, &sl.q_split, &sl.list_info,
                  &sl.list});
    free_pinned(sl.stage);
    for (auto &e : sl.ev)
        if (e) { (void)hipEventDestroy(e); e = nullptr; }
    if (sl.own_stream && sl.stream) (void)hipStreamDestroy(sl.stream);
    sl.stream = nullptr;
}

namespace {

// FP32 normalisation exactly as VectorMatrix::vectorNormalize
// (src/include/struct/VectorMatrix.hpp:51-66).  This file is compiled with
// -ffp-contract=off, so x*x is rounded before the add.
void normalize_rows(float *u, int64_t n, int32_t d, int64_t stride) {
#pragma omp parallel for schedule(static)
    for (int64_t i = 0; i < n; ++i) {
        float *row = u + i * stride;
        float l2 = 0.0f;
        for (int32_t j = 0; j < d; ++j) {
            const float sq = row[j] * row[j];
            l2 = l2 + sq;
        }
        l2 = std::sqrt(l2);
        if ((double)l2 <= 0.001) continue;
        for (int32_t j = 0; j < d; ++j) row[j] = row[j] / l2;
    }
}

bool ranks_valid(const int32_t *r, int32_t S, int64_t n_item) {
    if (S <= 0 || (int64_t)S >= n_item) return false;
    for (int32_t j = 0; j < S; ++j) {
        if (r[j] < 0 || (int64_t)r[j] >= n_item) return false;
        if (j > 0 && r[j] <= r[j - 1]) return false;
    }
    return true;
}

double ev_ms(hipEvent_t *ev, int a, int b) {
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, ev[a], ev[b]) != hipSuccess) return 0.0;
    return ms;
}

}  // namespace
}  // namespace rkr

using namespace rkr;

struct rkr_ctx : public rkr::Ctx {};

extern "C" {

const char *rkr_version(void) { return kVersion; }

int rkr_create(int device, size_t mem_budget_bytes, rkr_ctx **out) {
    if (!out) return RKR_ERR_INVALID;
    *out = nullptr;
    int n_dev = 0;
    if (hipGetDeviceCount(&n_dev) != hipSuccess || n_dev <= 0) return RKR_ERR_NODEVICE;
    if (device < 0 || device >= n_dev) return RKR_ERR_INVALID;
    if (hipSetDevice(device) != hipSuccess) return RKR_ERR_HIP;
    rkr_ctx *c = new (std::nothrow) rkr_ctx();
    if (!c) return RKR_ERR_NOMEM;
    c->device = device;
    size_t free_b = 0, total_b = 0;
    if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) { delete c; return RKR_ERR_HIP; }
    c->budget = mem_budget_bytes ? std::min(mem_budget_bytes, free_b) : (size_t)(0.9 * (double)free_b);
    int n_cu = 0;
    if (hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && n_cu > 0)
        c->n_cu = n_cu;
    int khz = 0;
    if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, device) == hipSuccess && khz > 0) c->clock_khz = khz;
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) { delete c; return RKR_ERR_HIP; }
    for (auto &e : c->ev)
        if (hipEventCreate(&e) != hipSuccess) { rkr_destroy(c); return RKR_ERR_HIP; }
    if (slot_init(c, c->main, false) != RKR_OK) { rkr_destroy(c); return RKR_ERR_HIP; }
    if (hipMalloc(&c->rho, 256) != hipSuccess) { c->rho = nullptr; rkr_destroy(c); return RKR_ERR_NOMEM; }
    // the no-allocation entry point's scratch: its address on this device,
    // looked up once per device (a failure is reported by that entry point)
    (void)noalloc_init(device);
    *out = c;
    return RKR_OK;
}

void rkr_destroy(rkr_ctx *c) {
    if (!c) return;
    (void)hipSetDevice(c->device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    free_scratch(c);
    slot_free(c, c->main);
    if (c->aux_ready) slot_free(c, c->aux);
    free_data(c);
    for (auto &e : c->ev)
        if (e) (void)hipEventDestroy(e);
    if (c->rho) (void)hipFree(c->rho);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
}

const char *rkr_last_error(const rkr_ctx *c) { return c ? c->err.c_str() : "null context"; }

int rkr_set_option(rkr_ctx *c, int option, int64_t value) {
    if (!c) return RKR_ERR_INVALID;
    switch (option) {
        case RKR_OPT_FORM:
            if (value != RKR_FORM_PLAIN && value != RKR_FORM_SCREENED)
                return set_err(c, RKR_ERR_INVALID, "unknown form");
            c->form = (int)value;
            return RKR_OK;
        case RKR_OPT_OUTPUT:
            if (value != RKR_OUTPUT_EXACT && value != RKR_OUTPUT_REFERENCE)
                return set_err(c, RKR_ERR_INVALID, "unknown output order");
            c->output = (int)value;
            return RKR_OK;
        case RKR_OPT_QUERY_BATCH:
            if (value < 0) return set_err(c, RKR_ERR_INVALID, "query batch must be >= 0");
            c->query_batch = value;
            return RKR_OK;
        case RKR_OPT_BUILD_BATCH:
            if (value < 0) return set_err(c, RKR_ERR_INVALID, "build batch must be >= 0");
            c->build_batch = value;
            return RKR_OK;
        case RKR_OPT_SCREEN_CHUNK:
            if (value < 0 || value > (1 << 30)) return set_err(c, RKR_ERR_INVALID, "screen chunk must be in [0, 2^30]");
            c->screen_chunk = (int32_t)value;
            return RKR_OK;
        case RKR_OPT_DENSE_TOP:
            if (value < 0 || value > 2) return set_err(c, RKR_ERR_INVALID, "dense top must be 0, 1 or 2");
            c->dense_top = (int)value;
            return RKR_OK;
        case RKR_OPT_SCREEN_ROWS:
            if (value != 0 && value != 32 && value != 64) return set_err(c, RKR_ERR_INVALID, "screen rows must be 0, 32 or 64");
            c->screen_rows = (int32_t)value;
            return RKR_OK;
        case RKR_OPT_DEDUP:
            if (value != 0 && value != 1) return set_err(c, RKR_ERR_INVALID, "dedup must be 0 or 1");
            c->dedup = (int)value;
            return RKR_OK;
        case RKR_OPT_COARSE:
            if (value != 0 && value != 1) return set_err(c, RKR_ERR_INVALID, "coarse must be 0 or 1");
            c->coarse = (int)value;
            return RKR_OK;
        case RKR_OPT_QUERY_SLOTS:
            if (value != 1 && value != 2) return set_err(c, RKR_ERR_INVALID, "query slots must be 1 or 2");
            c->query_slots = (int)value;
            return RKR_OK;
        case RKR_OPT_QSRP:
            if (value != 0 && value != 1) return set_err(c, RKR_ERR_INVALID, "qsrp must be 0 or 1");
            c->qsrp = (int)value;
            return RKR_OK;
        case kOptDpSpin:
            if (value < 0 || value > (1 << 20)) return set_err(c, RKR_ERR_INVALID, "DP looks must be in [0, 2^20]");
            c->dp_spin = (int32_t)value;
            return RKR_OK;
        default:
            return set_err(c, RKR_ERR_INVALID, "unknown option");
    }
}

int rkr_get_option(const rkr_ctx *c, int option, int64_t *value) {
    if (!c || !value) return RKR_ERR_INVALID;
    switch (option) {
        case RKR_OPT_FORM: *value = c->form; return RKR_OK;
        case RKR_OPT_OUTPUT: *value = c->output; return RKR_OK;
        case RKR_OPT_QUERY_BATCH: *value = c->query_batch; return RKR_OK;
        case RKR_OPT_BUILD_BATCH: *value = c->build_batch; return RKR_OK;
        case RKR_OPT_SCREEN_CHUNK: *value = c->screen_chunk; return RKR_OK;
        case RKR_OPT_DEDUP: *value = c->dedup; return RKR_OK;
        case RKR_OPT_SCREEN_ROWS: *value = c->screen_rows; return RKR_OK;
        case RKR_OPT_DENSE_TOP: *value = c->dense_top; return RKR_OK;
        case RKR_OPT_COARSE: *value = c->coarse; return RKR_OK;
        case RKR_OPT_QUERY_SLOTS: *value = c->query_slots; return RKR_OK;
        case RKR_OPT_QSRP: *value = c->qsrp; return RKR_OK;
        default: return RKR_ERR_INVALID;
    }
}

int rkr_sync(rkr_ctx *c) {
    if (!c) return RKR_ERR_INVALID;
    RKR_HIP(c, hipStreamSynchronize(c->stream));
    return RKR_OK;
}

int rkr_normalize_users(float *users, int64_t n_user, int32_t dim) {
    if (!users || n_user < 0 || dim <= 0) return RKR_ERR_INVALID;
    normalize_rows(users, n_user, dim, dim);
    return RKR_OK;
}

int rkr_uniform_sample_ranks(int64_t n_item, int32_t n_sample, int32_t *out) {
    // FindUniformSample, UniformSample.hpp:17-25
    if (!out || n_sample <= 0 || (int64_t)n_sample >= n_item) return RKR_ERR_INVALID;
    const int end_rank = (int)n_item - 1;
    const double delta = (end_rank - 0) * 1.0 / n_sample;
    for (int32_t j = 0; j < n_sample; ++j) out[j] = (int32_t)std::floor(j * delta);
    return RKR_OK;
}

int rkr_set_data(rkr_ctx *c, const float *users, int64_t n_user, const float *items, int64_t n_item, int32_t dim,
                 int normalize_users) {
    if (!c) return RKR_ERR_INVALID;
    if (!users || !items || n_user <= 0 || n_item <= 0 || dim <= 0)
        return set_err(c, RKR_ERR_INVALID, "set_data: empty or null input");
    if (n_user > INT32_MAX || n_item > INT32_MAX) return set_err(c, RKR_ERR_INVALID, "set_data: too many rows");
    if (dim > 4096) return set_err(c, RKR_ERR_INVALID, "set_data: dim > 4096 unsupported");
    {
        const double mu = max_abs(users, (size_t)n_user * dim), mp = max_abs(items, (size_t)n_item * dim);
        if (mu < 0 || mp < 0) return set_err(c, RKR_ERR_INVALID, "set_data: users and items must be finite");
        const double mu_n = normalize_users ? 1.0 : mu;  // normalised rows have |u_i| <= 1
        c->max_abs_user = mu_n;
        c->max_abs_item = mp;
        c->max_abs_user_raw = mu;
        if ((double)dim * mu_n * mp > kScoreLimit)
            return set_err(c, RKR_ERR_INVALID, "set_data: magnitudes would overflow FP32 scores");
    }
    RKR_HIP(c, hipSetDevice(c->device));
    RKR_HIP(c, hipStreamSynchronize(c->stream));
    free_scratch(c);
    free_data(c);
    const int32_t ld = padded_dim(dim);
    c->n_user = n_user;
    c->n_item = n_item;
    c->u_cap = n_user;
    c->i_cap = n_item;
    c->normalize_users = normalize_users != 0;
    c->dim = dim;
    c->ld = ld;
    // upload row-major with rows padded to ld floats (pad columns zero), users
    // normalised on the way
    auto upload = [&](const float *src, int64_t n, float **dst, bool normalize, const char *what) -> int {
        int rc = dev_alloc_t(c, dst, (size_t)n * ld, what);
        if (rc) return rc;
        const int64_t chunk = 65536;
        std::vector<float> tmp((size_t)std::min<int64_t>(chunk, n) * ld, 0.0f);
        for (int64_t r0 = 0; r0 < n; r0 += chunk) {
            const int64_t nr = std::min<int64_t>(chunk, n - r0);
            for (int64_t r = 0; r < nr; ++r)
                std::memcpy(&tmp[(size_t)r * ld], src + (size_t)(r0 + r) * dim, sizeof(float) * dim);
            if (normalize) normalize_rows(tmp.data(), nr, dim, ld);
            RKR_HIP(c, hipMemcpy(*dst + r0 * ld, tmp.data(), sizeof(float) * (size_t)nr * ld, hipMemcpyHostToDevice));
        }
        return RKR_OK;
    };
    int rc = upload(users, n_user, &c->users, normalize_users != 0, "users");
    if (rc) { free_data(c); return rc; }
    rc = upload(items, n_item, &c->items, false, "items");
    if (rc) { free_data(c); return rc; }
    rc = dev_alloc_t(c, &c->usersT, (size_t)((n_user + 63) / 64) * 64 * ld, "user panels");
    if (rc) { free_data(c); return rc; }
    RKR_HIP(c, launch_make_panels(c->stream, c->users, n_user, ld, c->usersT));
    // screened form: hi/lo BF16 item rows and norm bounds (d <= 256)
    const int32_t kp = (dim + 31) / 32 * 32;
    if (kp <= screen_max_kp()) {
        c->kp = kp;
        // |s^ - s| <= C ||u|| ||p|| + abs: dropped split terms (3.2 * 2^-16),
        // FP32 accumulation of 3*kp exact products at <= 2^-23 each (x1.03 for
        // the split magnitudes), the sequential rule's own rounding
        // (gamma_dim at 2^-24), times a 1% margin that also absorbs the FP32
        // evaluation of the bound itself.
        const double n3 = 3.0 * kp, e23 = std::ldexp(1.0, -23), e24 = std::ldexp(1.0, -24);
        const double g_mfma = n3 * e23 / (1.0 - n3 * e23), g_rule = dim * e24 / (1.0 - dim * e24);
        const double C = (3.2 * std::ldexp(1.0, -16) + 1.03 * g_mfma + g_rule) * 1.01;
        c->screen_C = std::nextafter((float)C, INFINITY);
        // the coarse first pass's single product u_hi q_hi: its error scale
        // per query (k_prep_items) takes the users' largest BF16 residual
        // ratio rho (k_user_norms), the FP32 accumulation of kp exact
        // products and the rule's own rounding
        const double n1 = (double)kp;
        c->coarse_g1 = n1 * e23 / (1.0 - n1 * e23);
        c->coarse_grule = g_rule;
        c->screen_abs = screen_abs_floor(kp, c->max_abs_user, c->max_abs_item);
        if ((rc = dev_alloc_t(c, &c->item_hi, (size_t)n_item * kp, "item hi")) ||
            (rc = dev_alloc_t(c, &c->item_lo, (size_t)n_item * kp, "item lo")) ||
            (rc = dev_alloc_t(c, &c->item_norm, (size_t)n_item, "item norms")) ||
            (rc = dev_alloc_t(c, &c->user_norm, (size_t)n_user, "user norms")) ||
            (rc = dev_alloc_t(c, &c->user_hi, (size_t)n_user * kp, "user hi")) ||
            (rc = dev_alloc_t(c, &c->user_lo, (size_t)n_user * kp, "user lo"))) {
            free_data(c);
            return rc;
        }
        RKR_HIP(c, launch_prep_items(c->stream, c->items, n_item, ld, dim, kp, c->item_hi, c->item_lo, c->item_norm));
        RKR_HIP(c, hipMemsetAsync(c->rho, 0, sizeof(float), c->stream));
        RKR_HIP(c, launch_user_norms(c->stream, c->users, n_user, ld, dim, c->user_norm, c->rho));
        RKR_HIP(c, launch_prep_items(c->stream, c->users, n_user, ld, dim, kp, c->user_hi, c->user_lo, nullptr));
    }
    c->items_base = c->items;
    c->n_item_base = n_item;
    RKR_HIP(c, hipStreamSynchronize(c->stream));
    return RKR_OK;
}

int rkr_build_table(rkr_ctx *c, const int32_t *ranks, int32_t S, double *build_ms) {
    if (!c) return RKR_ERR_INVALID;
    return rkr::build_table(c, ranks, S, build_ms, false);
}

}  // extern "C"

namespace rkr {

int rebuild_table(Ctx *c) {
    if (!c->table) return set_err(c, RKR_ERR_STATE, "rebuild: no table");
    std::vector<int32_t> ranks((size_t)c->n_sample);
    const int rc = rkr_uniform_sample_ranks(c->n_item, c->n_sample, ranks.data());
    if (rc) return set_err(c, rc, "rebuild: n_sample does not fit the current items");
    return build_table(c, ranks.data(), c->n_sample, nullptr, true);
}

int build_table(Ctx *c, const int32_t *ranks, int32_t S, double *build_ms, bool keep_update_buffers) {
    if (!c->users) return set_err(c, RKR_ERR_STATE, "build_table: no data");
    if (!ranks || S > kMaxSample || !ranks_valid(ranks, S, c->n_item))
        return set_err(c, RKR_ERR_INVALID, "build_table: ranks must be strictly increasing in [0, n_item), "
                                           "0 < n_sample < n_item, n_sample <= " + std::to_string(kMaxSample));
    RKR_HIP(c, hipSetDevice(c->device));
    RKR_HIP(c, hipStreamSynchronize(c->stream));
    const int64_t cap = std::max(c->u_cap, c->n_user);
    std::vector<int32_t> hr(ranks, ranks + S), hq;
    if (c->dense_top) hq = query_table_ranks(hr, c->n_item, c->dense_top);
    const int32_t nqs = (int32_t)hq.size() > S ? (int32_t)hq.size() : 0;
    // buffers of the last table that have the new one's size are used again,
    // unless a batch may be reading them (six allocations and as many frees:
    // 5752 users x 5201 items 1.6 -> 1.16 ms, 100k x 6001 14.6 -> 13.5)
    const size_t n_ranks = sizeof(int32_t) * S, n_qr = sizeof(int32_t) * nqs, row = sizeof(float) * (size_t)cap;
    int32_t *k_ranks = keep_buffer(c, c->ranks, n_ranks), *k_qranks = keep_buffer(c, c->qranks, n_qr);
    int32_t *k_qcol = nqs ? keep_buffer(c, c->qcol, n_ranks) : nullptr;
    float *k_table = keep_buffer(c, c->table, row * S), *k_qtable = keep_buffer(c, c->qtable, row * nqs);
    float *k_guards = keep_buffer(c, c->gvals, guard_bytes(cap, true));
    free_table(c);
    free_update_state(c, keep_update_buffers);  // the new table describes the current item set
    c->ranks = k_ranks;
    c->qranks = k_qranks;
    c->qcol = k_qcol;
    c->table = k_table;
    c->qtable = k_qtable;
    if (k_guards) place_guards(c, Guards{k_guards, cap, true});
    int rc = RKR_OK;
    if ((!c->ranks && (rc = dev_alloc_t(c, &c->ranks, (size_t)S, "ranks"))) ||
        (!c->table && (rc = dev_alloc_t(c, &c->table, (size_t)cap * S, "table"))) ||
        (nqs && !c->qranks && (rc = dev_alloc_t(c, &c->qranks, (size_t)nqs, "query table ranks"))) ||
        (nqs && !c->qcol && (rc = dev_alloc_t(c, &c->qcol, (size_t)S, "query table columns"))) ||
        (nqs && !c->qtable && (rc = dev_alloc_t(c, &c->qtable, (size_t)cap * nqs, "query table"))) ||
        // beside them the smallest score block fits: two rows of the free budget
        (!c->gvals && (rc = alloc_guards(c, cap, 2 * sizeof(float) * (size_t)c->n_item)))) {
        free_table(c);
        return rc;
    }
    c->n_sample = S;
    c->h_ranks.swap(hr);
    RKR_HIP(c, hipMemcpyAsync(c->ranks, ranks, sizeof(int32_t) * S, hipMemcpyHostToDevice, c->stream));
    if (nqs) {
        // the query table: select at its ranks, then copy the sampled columns
        c->h_qranks.swap(hq);
        std::vector<int32_t> col((size_t)S);
        for (int32_t j = 0, q = 0; j < S; ++j) {
            while (c->h_qranks[q] != ranks[j]) ++q;
            col[j] = q;
        }
        c->n_qs = nqs;
        RKR_HIP(c, hipMemcpyAsync(c->qranks, c->h_qranks.data(), sizeof(int32_t) * nqs, hipMemcpyHostToDevice,
                                  c->stream));
        RKR_HIP(c, hipMemcpyAsync(c->qcol, col.data(), sizeof(int32_t) * S, hipMemcpyHostToDevice, c->stream));
        RKR_HIP(c, hipStreamSynchronize(c->stream));
    }

    set_table_columns(c);

    // user batch: the score block [nb x n_item] lives in HBM between the
    // GEMM and the selection; size it from the remaining budget (the
    // reference sizes its batch from free memory the same way,
    // GPUComputeSort.hpp:112-135).
    const size_t row_bytes = sizeof(float) * (size_t)c->n_item;
    const size_t avail = free_bytes(c);
    const MiscUse use(c);
    int64_t nb = (int64_t)std::min<size_t>(avail / 2 / row_bytes, (size_t)(8ull << 30) / row_bytes);
    if (c->build_batch > 0) nb = std::min<int64_t>(nb, c->build_batch);
    nb = std::min<int64_t>(nb, c->n_user);
    if (nb > 128) nb = nb / 128 * 128;
    if (nb <= 0) { free_table(c); return set_err(c, RKR_ERR_NOMEM, "build_table: no memory for a score block"); }
    DeviceBuf &blk = c->misc;
    rc = ensure(c, blk, (size_t)nb * row_bytes, "score block");
    if (rc) { free_table(c); return rc; }
    float *scores = reinterpret_cast<float *>(blk.p);
    RKR_HIP(c, hipEventRecord(c->ev[0], c->stream));
    for (int64_t u0 = 0; u0 < c->n_user; u0 += nb) {
        const int64_t n = std::min<int64_t>(nb, c->n_user - u0);
        RKR_HIP(c, launch_scores_store(c->stream, c->users + u0 * c->ld, n, c->ld, c->items, c->n_item, c->ld,
                                       c->dim, scores, c->n_item, true));
        if (c->qtable) {
            RKR_HIP(c, launch_select_rows(c->stream, scores, n, c->n_item, c->qranks, c->n_qs,
                                          c->qtable + u0 * c->n_qs));
            RKR_HIP(c, launch_gather_cols(c->stream, c->qtable + u0 * c->n_qs, c->n_qs, c->qcol, S, n,
                                          c->table + u0 * S, S));
        } else {
            RKR_HIP(c, launch_select_rows(c->stream, scores, n, c->n_item, c->ranks, S, c->table + u0 * S));
        }
    }
    if ((rc = refresh_guard_values(c, 0, c->n_user))) { free_table(c); return rc; }
    RKR_HIP(c, hipEventRecord(c->ev[1], c->stream));
    RKR_HIP(c, hipStreamSynchronize(c->stream));
    if (build_ms) *build_ms = ev_ms(c->ev, 0, 1);
    return RKR_OK;
}

}  // namespace rkr

extern "C" {

int rkr_set_table(rkr_ctx *c, const int32_t *ranks, int32_t S, const float *table, float eps) {
    if (!c) return RKR_ERR_INVALID;
    if (!c->users) return set_err(c, RKR_ERR_STATE, "set_table: no data");
    if (!ranks || !table || S > kMaxSample || !ranks_valid(ranks, S, c->n_item))
        return set_err(c, RKR_ERR_INVALID, "set_table: bad ranks");
    if (!(eps >= 0.0f) || std::isinf(eps)) return set_err(c, RKR_ERR_INVALID, "set_table: eps must be finite, >= 0");
    RKR_HIP(c, hipSetDevice(c->device));
    RKR_HIP(c, hipStreamSynchronize(c->stream));
    free_table(c);
    free_update_state(c);  // the installed table describes the current item set
    int rc = dev_alloc_t(c, &c->ranks, (size_t)S, "ranks");
    if (rc) return rc;
    rc = dev_alloc_t(c, &c->table, (size_t)std::max(c->u_cap, c->n_user) * S, "table");
    if (!rc) rc = alloc_guards(c, std::max(c->u_cap, c->n_user), 0);
    if (rc) { free_table(c); return rc; }
    c->n_sample = S;
    c->h_ranks.assign(ranks, ranks + S);
    c->table_eps = eps;
    set_table_columns(c);
    RKR_HIP(c, hipMemcpy(c->ranks, ranks, sizeof(int32_t) * S, hipMemcpyHostToDevice));
    RKR_HIP(c, hipMemcpy(c->table, table, sizeof(float) * (size_t)c->n_user * S, hipMemcpyHostToDevice));
    if ((rc = refresh_guard_values(c, 0, c->n_user))) { free_table(c); return rc; }
    RKR_HIP(c, hipStreamSynchronize(c->stream));
    return RKR_OK;
}

extern "C++" {
namespace {
// A device allocation freed when the scope ends.
struct ScopedDev {
    rkr::Ctx *c;
    void *p = nullptr;
    size_t bytes = 0;
    int alloc(size_t n, const char *what) {
        rkr::dev_free(c, p, bytes);
        p = nullptr;
        bytes = n;
        return rkr::dev_alloc(c, &p, n, what);
    }
    template <class T>
    T *as() const { return static_cast<T *>(p); }
    ~ScopedDev() { rkr::dev_free(c, p, bytes); }
};

// Runs fn(i0, i1) over [0, n) in up to 16 ranges, one host thread per range and
// no range under min_per units; a range whose thread cannot start runs here.
template <class F>
void host_ranges(int64_t n, int64_t min_per, F &&fn) {
    if (n <= 0) return;
    const int64_t nt = std::min<int64_t>({(int64_t)std::max(1u, std::thread::hardware_concurrency()), 16,
                                          std::max<int64_t>(1, n / std::max<int64_t>(1, min_per))});
    std::vector<std::thread> th;
    int64_t launched = 1;
    try {
        th.reserve((size_t)nt);
        for (; launched < nt; ++launched) th.emplace_back(fn, n * launched / nt, n * (launched + 1) / nt);
    } catch (...) {
    }
    fn(0, n / nt);
    for (int64_t t = launched; t < nt; ++t) fn(n * t / nt, n * (t + 1) / nt);
    for (auto &x : th) x.join();
}

// Device-to-host copies through two pinned staging buffers: while one chunk
// crosses the link, the host consumes the previous one.  A plain copy into
// pageable memory runs at a fraction of the link's rate.
constexpr size_t kStageBytes = (size_t)32 << 20;
struct Staging {
    hipStream_t s;
    size_t chunk = 0;
    void *p[2] = {nullptr, nullptr};
    hipEvent_t e[2] = {nullptr, nullptr};
    explicit Staging(hipStream_t st) : s(st) {}
    Staging(const Staging &) = delete;
    Staging &operator=(const Staging &) = delete;
    ~Staging() {
        (void)hipStreamSynchronize(s);  // no copy into a buffer outlives it
        for (int k = 0; k < 2; ++k) {
            if (p[k]) {
                if (pinned) (void)hipHostFree(p[k]);
                else std::free(p[k]);
            }
            if (e[k]) (void)hipEventDestroy(e[k]);
        }
    }
    bool pinned = true;
    // Pinned buffers when the runtime grants them; otherwise ordinary pageable
    // buffers, which the same asynchronous copies fill at the pageable rate.
    hipError_t init(size_t bytes) {
        chunk = std::max<size_t>(bytes, 1);
        for (int k = 0; k < 2 && pinned; ++k)
            if (hipHostMalloc(&p[k], chunk, hipHostMallocDefault) != hipSuccess) {
                (void)hipGetLastError();
                for (int j = 0; j < k; ++j) (void)hipHostFree(p[j]);
                p[0] = p[1] = nullptr;
                pinned = false;
            }
        for (int k = 0; k < 2; ++k) {
            if (!pinned && !(p[k] = std::malloc(chunk))) return hipErrorOutOfMemory;
            const hipError_t r = hipEventCreateWithFlags(&e[k], hipEventDisableTiming);
            if (r != hipSuccess) return r;
        }
        return hipSuccess;
    }
    // Chunk k of n_chunk: issue(k, buf) enqueues its copy into buf on the stream
    // (at most `chunk` bytes); take(k, buf) consumes it once it has arrived and
    // returns false to stop.
    template <class Issue, class Take>
    hipError_t run(int64_t n_chunk, Issue &&issue, Take &&take) {
        auto put = [&](int64_t k) {
            const hipError_t r = issue(k, p[k & 1]);
            return r == hipSuccess ? hipEventRecord(e[k & 1], s) : r;
        };
        hipError_t r = n_chunk > 0 ? put(0) : hipSuccess;
        if (r == hipSuccess && n_chunk > 1) r = put(1);
        for (int64_t k = 0; r == hipSuccess && k < n_chunk; ++k) {
            r = hipEventSynchronize(e[k & 1]);
            if (r != hipSuccess || !take(k, static_cast<const char *>(p[k & 1]))) break;
            if (k + 2 < n_chunk) r = put(k + 2);  // the buffer just consumed takes the chunk after next
        }
        return r;
    }
    // dst[0, bytes) = src[0, bytes), src in device memory; host threads copy out.
    hipError_t to_host(void *dst, const void *src, size_t bytes) {
        const int64_t n_chunk = (int64_t)((bytes + chunk - 1) / chunk);
        return run(
            n_chunk,
            [&](int64_t k, void *buf) {
                const size_t off = (size_t)k * chunk, len = std::min(chunk, bytes - off);
                return hipMemcpyAsync(buf, static_cast<const char *>(src) + off, len, hipMemcpyDeviceToHost, s);
            },
            [&](int64_t k, const char *buf) {
                const size_t off = (size_t)k * chunk, len = std::min(chunk, bytes - off);
                char *d = static_cast<char *>(dst) + off;
                host_ranges((int64_t)len, (int64_t)1 << 20,
                            [d, buf](int64_t a, int64_t b) { std::memcpy(d + a, buf + a, (size_t)(b - a)); });
                return true;
            });
    }
};
}  // namespace

// Calls sink(rows, user, m, more, spare) for users [u0, u0 + n) in batches of m
// rows: rows (device memory, stride n_item) holds each user's scores against the
// current items, sorted in descending order, more is scratch of `extra` floats
// per row, and spare of `wish` floats per row behind it, null where they do not
// fit beside one row.  The block size follows the memory budget as the table
// build's does.
template <class Sink>
static int sorted_score_batches(rkr_ctx *c, int64_t u0, int64_t n, const char *what, Sink &&sink,
                                double *gemm_ms = nullptr, double *sort_ms = nullptr, int64_t extra = 0,
                                int64_t wish = 0) {
    const int64_t I = c->n_item;
    const size_t row_bytes = sizeof(float) * (size_t)I;
    // the scratch kept from an earlier call is there to be used
    const size_t avail = free_bytes(c);
    const MiscUse use(c);
    int64_t nb = (int64_t)std::min<size_t>(avail / 3 / row_bytes, (size_t)(2ull << 30) / row_bytes);
    if (c->build_batch > 0) nb = std::min<int64_t>(nb, c->build_batch);
    nb = std::min<int64_t>(nb, n);
    // a third of the budget for the block; its sort scratch and the caller's floats
    // are as much again for each of nb rows, but not more than all of it
    const auto need = [&](int64_t rows, int64_t per_row) { return (size_t)rows * (2 * row_bytes + sizeof(float) * (size_t)per_row) + 512; };
    if (wish > 0 && need(1, extra + wish) > avail) wish = 0;
    while (nb > 1 && need(nb, extra + wish) > avail) nb -= std::max<int64_t>(1, nb / 16);
    if (nb <= 0) return set_err(c, RKR_ERR_NOMEM, std::string(what) + ": no memory for a score block");
    // the build scratch, kept between calls (allocating and freeing the block
    // took 1 ms of a call over 13k users)
    const int64_t tmp_rows = std::min<int64_t>(nb, sort_rows_in_flight(I, c->n_cu));
    const size_t blk_bytes = ((size_t)nb * row_bytes + 255) & ~(size_t)255;
    const size_t tmp_bytes = ((size_t)tmp_rows * row_bytes + 255) & ~(size_t)255;
    int rc = ensure(c, c->misc, blk_bytes + tmp_bytes + sizeof(float) * (size_t)(nb * (extra + wish)), "score block");
    if (rc) return rc;
    char *buf = reinterpret_cast<char *>(c->misc.p);
    float *blk = reinterpret_cast<float *>(buf), *tmp = reinterpret_cast<float *>(buf + blk_bytes);
    float *more = reinterpret_cast<float *>(buf + blk_bytes + tmp_bytes);
    float *spare = wish > 0 ? more + nb * extra : nullptr;
    for (int64_t b0 = 0; b0 < n; b0 += nb) {
        const int64_t m = std::min<int64_t>(nb, n - b0);
        RKR_HIP(c, hipEventRecord(c->ev[0], c->stream));
        RKR_HIP(c, launch_scores_store(c->stream, c->users + (u0 + b0) * c->ld, m, c->ld, c->items, I, c->ld,
                                       c->dim, blk, I, true));
        RKR_HIP(c, hipEventRecord(c->ev[1], c->stream));
        RKR_HIP(c, launch_sort_rows(c->stream, blk, I, m, I, blk, tmp, tmp_rows, I, c->n_cu));
        RKR_HIP(c, hipEventRecord(c->ev[2], c->stream));
        if ((rc = sink(blk, u0 + b0, m, more, spare))) return rc;  // the sink synchronises the stream
        if (gemm_ms) *gemm_ms += ev_ms(c->ev, 0, 1);
        if (sort_ms) *sort_ms += ev_ms(c->ev, 1, 2);
    }
    return RKR_OK;
}
}  // extern "C++"

int rkr_get_table(rkr_ctx *c, int64_t user_begin, int64_t n_rows, float *out) {
    if (!c || !out) return RKR_ERR_INVALID;
    if (!c->table) return set_err(c, RKR_ERR_STATE, "get_table: no table");
    if (user_begin < 0 || n_rows < 0 || user_begin + n_rows > c->n_user)
        return set_err(c, RKR_ERR_INVALID, "get_table: row range out of bounds");
    if (n_rows == 0) return RKR_OK;
    RKR_HIP(c, hipSetDevice(c->device));
    RKR_HIP(c, hipStreamSynchronize(c->stream));
    const size_t bytes = sizeof(float) * (size_t)n_rows * c->n_sample;
    Staging stg{c->stream};
    RKR_HIP(c, stg.init(std::min(kStageBytes, bytes)));
    RKR_HIP(c, stg.to_host(out, c->table + user_begin * c->n_sample, bytes));
    return RKR_OK;
}

int rkr_sorted_scores(rkr_ctx *c, int64_t user_begin, int64_t n_rows, float *out) {
    // ComputeScoreTableBatch::ComputeSortItemsBatch (ComputeScoreTableBatch.hpp:79-92)
    if (!c || (n_rows > 0 && !out)) return c ? set_err(c, RKR_ERR_INVALID, "sorted_scores: bad arguments") : RKR_ERR_INVALID;
    if (!c->users) return set_err(c, RKR_ERR_STATE, "sorted_scores: no data");
    if (user_begin < 0 || n_rows < 0 || user_begin + n_rows > c->n_user)
        return set_err(c, RKR_ERR_INVALID, "sorted_scores: row range out of bounds");
    if (n_rows == 0) return RKR_OK;
    RKR_HIP(c, hipSetDevice(c->device));
    RKR_HIP(c, hipStreamSynchronize(c->stream));
    const int64_t I = c->n_item;
    Staging stg{c->stream};
    RKR_HIP(c, stg.init(std::min(kStageBytes, sizeof(float) * (size_t)(n_rows * I))));
    return sorted_score_batches(c, user_begin, n_rows, "sorted_scores", [&](const float *rows, int64_t u, int64_t m, float *, float *) {
        RKR_HIP(c, stg.to_host(out + (u - user_begin) * I, rows, sizeof(float) * (size_t)(m * I)));
        return (int)RKR_OK;
    });
}

int rkr_save_score_table(rkr_ctx *c, const char *path, int64_t n_rows, double *timing_ms) {
    // ReadAll::BuildIndexLoop layout (ReadAll.hpp:80-87) as BuildScoreTableBatch.cpp:69-144 writes it
    if (!c || !path) return c ? set_err(c, RKR_ERR_INVALID, "save_score_table: bad arguments") : RKR_ERR_INVALID;
    if (!c->users) return set_err(c, RKR_ERR_STATE, "save_score_table: no data");
    if (n_rows < 0) n_rows = c->n_user;
    if (n_rows > c->n_user) return set_err(c, RKR_ERR_INVALID, "save_score_table: more rows than users");
    RKR_HIP(c, hipSetDevice(c->device));
    RKR_HIP(c, hipStreamSynchronize(c->stream));
    const int64_t I = c->n_item;
    // the file is written straight from the pinned staging buffers, one chunk
    // while the next crosses the link
    Staging stg{c->stream};
    RKR_HIP(c, stg.init(std::min(kStageBytes, sizeof(float) * (size_t)(n_rows * I))));
    FILE *f = std::fopen(path, "wb");
    if (!f) return set_err(c, RKR_ERR_IO, std::string("save_score_table: cannot open ") + path);
    double gemm_ms = 0, sort_ms = 0, write_s = 0;
    const double t0 = rkr_now();
    int rc = n_rows == 0 ? (int)RKR_OK
                         : sorted_score_batches(c, 0, n_rows, "save_score_table",
                                                [&](const float *rows, int64_t, int64_t m, float *, float *) {
        const size_t bytes = sizeof(float) * (size_t)(m * I);
        bool ok = true;
        RKR_HIP(c, stg.run(
                       (int64_t)((bytes + stg.chunk - 1) / stg.chunk),
                       [&](int64_t k, void *buf) {
                           const size_t off = (size_t)k * stg.chunk, len = std::min(stg.chunk, bytes - off);
                           return hipMemcpyAsync(buf, reinterpret_cast<const char *>(rows) + off, len,
                                                 hipMemcpyDeviceToHost, c->stream);
                       },
                       [&](int64_t k, const char *buf) {
                           const size_t off = (size_t)k * stg.chunk, len = std::min(stg.chunk, bytes - off);
                           const double w0 = rkr_now();
                           ok = std::fwrite(buf, 1, len, f) == len;
                           write_s += rkr_now() - w0;
                           return ok;
                       }));
        if (!ok) return set_err(c, RKR_ERR_IO, std::string("save_score_table: write failed on ") + path);
        return (int)RKR_OK;
    }, &gemm_ms, &sort_ms);
    const double w0 = rkr_now();
    if (std::fclose(f) != 0 && !rc) rc = set_err(c, RKR_ERR_IO, std::string("save_score_table: close failed on ") + path);
    write_s += rkr_now() - w0;
    if (timing_ms) {
        timing_ms[0] = gemm_ms;
        timing_ms[1] = sort_ms;
        timing_ms[2] = (rkr_now() - t0 - write_s) * 1e3;
        timing_ms[3] = write_s * 1e3;
    }
    return rc;
}

int rkr_query_rank_distribution(rkr_ctx *c, const int32_t *item_ids, int32_t n_sample_item, int32_t *accu,
                                double *device_ms) {
    // ComputeQueryRankByComputation (src/app/build-index/QueryRankByComputation.hpp:122-242): for every sample
    // item s and user u, rank(u, s) = #{items scoring above <u, s>}, the lower_bound with greater<float> in
    // u's sorted row (QueryRankGPU.hpp:63-92); accu[s][r] = #{u : rank(u, s) <= r}, r = 0..n_item.
    if (!c || !item_ids || !accu || n_sample_item <= 0)
        return c ? set_err(c, RKR_ERR_INVALID, "query_rank_distribution: bad arguments") : RKR_ERR_INVALID;
    if (!c->users) return set_err(c, RKR_ERR_STATE, "query_rank_distribution: no data");
    const int64_t I = c->n_item, W = I + 1, ns = n_sample_item;
    std::vector<int64_t> ids((size_t)ns);
    for (int64_t s = 0; s < ns; ++s) {
        if (item_ids[s] < 0 || item_ids[s] >= I) return set_err(c, RKR_ERR_INVALID, "query_rank_distribution: bad item id");
        ids[s] = item_ids[s];
    }
    RKR_HIP(c, hipSetDevice(c->device));
    RKR_HIP(c, hipStreamSynchronize(c->stream));
    ScopedDev smat{c}, dids{c}, hist{c};
    int rc = smat.alloc(sizeof(float) * (size_t)(ns * c->ld), "sample items");
    if (!rc) rc = dids.alloc(sizeof(int64_t) * (size_t)ns, "sample ids");
    if (!rc) rc = hist.alloc(sizeof(int32_t) * (size_t)(ns * W), "rank histogram");
    if (rc) return rc;
    int32_t *h = hist.as<int32_t>();
    RKR_HIP(c, hipMemcpyAsync(dids.p, ids.data(), dids.bytes, hipMemcpyHostToDevice, c->stream));
    RKR_HIP(c, hipMemsetAsync(hist.p, 0, hist.bytes, c->stream));
    RKR_HIP(c, launch_gather_rows(c->stream, c->items, c->ld, dids.as<const int64_t>(), ns, c->ld, smat.as<float>(),
                                  c->ld));
    double ms = 0;
    rc = sorted_score_batches(c, 0, c->n_user, "query_rank_distribution", [&](const float *rows, int64_t u, int64_t m, float *qbuf, float *rbuf) {
        RKR_HIP(c, hipEventRecord(c->ev[3], c->stream));
        RKR_HIP(c, launch_scores_store(c->stream, c->users + u * c->ld, m, c->ld, smat.as<float>(), ns, c->ld,
                                       c->dim, qbuf, ns, true));
        RKR_HIP(c, launch_rank_hist(c->stream, rows, I, m, I, qbuf, ns, (int32_t)ns, h, reinterpret_cast<uint16_t *>(rbuf)));
        RKR_HIP(c, hipEventRecord(c->ev[4], c->stream));
        RKR_HIP(c, hipEventSynchronize(c->ev[4]));
        ms += ev_ms(c->ev, 0, 2) + ev_ms(c->ev, 3, 4);
        return (int)RKR_OK;
    }, nullptr, nullptr, ns + (ns & 1), rank_row(ns) / 2);  // a batch's scores (8-byte aligned ends) and, if they fit, 16-bit ranks
    if (rc) return rc;
    // The counts leave through the pinned staging buffers in chunks of whole
    // rows; host threads turn each chunk's counts per rank into users with
    // rank <= r, written into the caller's rows, while the next chunk copies.
    const int64_t chunk_rows = std::min<int64_t>(ns, std::max<int64_t>(1, (int64_t)(kStageBytes / sizeof(int32_t)) / W));
    Staging stg{c->stream};
    RKR_HIP(c, stg.init(sizeof(int32_t) * (size_t)(chunk_rows * W)));
    RKR_HIP(c, stg.run(
                   (ns + chunk_rows - 1) / chunk_rows,
                   [&](int64_t k, void *buf) {
                       const int64_t r0 = k * chunk_rows, nr = std::min(chunk_rows, ns - r0);
                       return hipMemcpyAsync(buf, h + r0 * W, sizeof(int32_t) * (size_t)(nr * W),
                                             hipMemcpyDeviceToHost, c->stream);
                   },
                   [&](int64_t k, const char *buf) {
                       const int64_t r0 = k * chunk_rows, nr = std::min(chunk_rows, ns - r0);
                       const int32_t *src = reinterpret_cast<const int32_t *>(buf);
                       host_ranges(nr, std::max<int64_t>(1, ((int64_t)1 << 16) / W), [src, accu, r0, W](int64_t s0, int64_t s1) {
                           for (int64_t s = s0; s < s1; ++s) {
                               const int32_t *x = src + s * W;
                               int32_t *row = accu + (r0 + s) * W;
                               int32_t run = 0;
                               for (int64_t r = 0; r < W; ++r) row[r] = run += x[r];
                           }
                       });
                       return true;
                   }));
    if (device_ms) *device_ms = ms;
    return RKR_OK;
}

int rkr_get_ranks(const rkr_ctx *c, int32_t *out, int32_t *n_sample) {
    if (!c) return RKR_ERR_INVALID;
    if (n_sample) *n_sample = c->n_sample;
    if (out && c->n_sample) std::memcpy(out, c->h_ranks.data(), sizeof(int32_t) * c->n_sample);
    return RKR_OK;
}

int rkr_save_table(rkr_ctx *c, const char *path) {
    // SampleSearch::SaveIndex layout (SampleSearch.hpp:186-194)
    if (!c || !path) return RKR_ERR_INVALID;
    if (!c->table) return set_err(c, RKR_ERR_STATE, "save_table: no table");
    // The table describes the item set it was built from; with pending inserts
    // or deletes a saved file would pair those rows with the current n_item and
    // lose the updates' rank offsets when it is loaded back.
    if (c->n_ins > 0 || c->n_del > 0)
        return set_err(c, RKR_ERR_STATE,
                       "save_table: item updates are pending; rebuild the table (rkr_build_table) before saving");
    RKR_HIP(c, hipSetDevice(c->device));
    RKR_HIP(c, hipStreamSynchronize(c->stream));
    // the table is written straight from the pinned staging buffers, one chunk
    // while the next crosses the link
    const size_t bytes = sizeof(float) * (size_t)c->n_user * c->n_sample;
    Staging stg{c->stream};
    RKR_HIP(c, stg.init(std::min(kStageBytes, std::max<size_t>(bytes, 1))));
    FILE *f = std::fopen(path, "wb");
    if (!f) return set_err(c, RKR_ERR_IO, std::string("save_table: cannot open ") + path);
    const size_t hdr[3] = {(size_t)c->n_sample, (size_t)c->n_item, (size_t)c->n_user};
    bool ok = std::fwrite(hdr, sizeof(size_t), 3, f) == 3;
    ok = ok && std::fwrite(c->h_ranks.data(), sizeof(int32_t), c->n_sample, f) == (size_t)c->n_sample;
    const hipError_t e = !ok ? hipSuccess : stg.run(
        (int64_t)((bytes + stg.chunk - 1) / stg.chunk),
        [&](int64_t k, void *buf) {
            const size_t off = (size_t)k * stg.chunk, len = std::min(stg.chunk, bytes - off);
            return hipMemcpyAsync(buf, reinterpret_cast<const char *>(c->table) + off, len, hipMemcpyDeviceToHost,
                                  c->stream);
        },
        [&](int64_t k, const char *buf) {
            const size_t off = (size_t)k * stg.chunk, len = std::min(stg.chunk, bytes - off);
            return ok = std::fwrite(buf, 1, len, f) == len;
        });
    ok = (std::fclose(f) == 0) && ok;
    if (e != hipSuccess) return set_err(c, RKR_ERR_HIP, std::string("save_table: ") + hipGetErrorString(e));
    if (!ok) return set_err(c, RKR_ERR_IO, std::string("save_table: short write to ") + path);
    return RKR_OK;
}

int rkr_load_table(rkr_ctx *c, const char *path, float eps) {
    // SampleSearch::LoadIndex layout (SampleSearch.hpp:229-241)
    if (!c || !path) return RKR_ERR_INVALID;
    if (!c->users) return set_err(c, RKR_ERR_STATE, "load_table: no data");
    FILE *f = std::fopen(path, "rb");
    if (!f) return set_err(c, RKR_ERR_IO, std::string("load_table: cannot open ") + path);
    size_t hdr[3];
    if (std::fread(hdr, sizeof(size_t), 3, f) != 3) { std::fclose(f); return set_err(c, RKR_ERR_IO, "load_table: short header"); }
    const size_t S = hdr[0], I = hdr[1], U = hdr[2];
    if ((int64_t)I != c->n_item || (int64_t)U != c->n_user || S == 0 || S > (size_t)kMaxSample) {
        std::fclose(f);
        return set_err(c, RKR_ERR_IO, "load_table: header (n_sample " + std::to_string(S) + ", n_item " +
                                          std::to_string(I) + ", n_user " + std::to_string(U) +
                                          ") does not match the data");
    }
    std::vector<int32_t> r(S);
    std::vector<float> t(S * U);
    bool ok = std::fread(r.data(), sizeof(int32_t), S, f) == S;
    ok = ok && std::fread(t.data(), sizeof(float), t.size(), f) == t.size();
    std::fclose(f);
    if (!ok) return set_err(c, RKR_ERR_IO, "load_table: file too short");
    return rkr_set_table(c, r.data(), (int32_t)S, t.data(), eps);
}

int64_t rkr_index_size_bytes(const rkr_ctx *c) {
    if (!c) return 0;
    return (int64_t)sizeof(int32_t) * c->n_sample + (int64_t)sizeof(float) * c->n_user * c->n_sample;
}

int32_t rkr_query_table_cols(const rkr_ctx *c) { return c && c->qtable ? c->n_qs : 0; }

}  // extern "C"

namespace {

constexpr int32_t kSplitMinQueries = 512;

// Answers queries [0, n) on the main slot, or -- with two query slots, at
// least kSplitMinQueries queries and two or more device batches -- the first
// half of the batches on the main slot and the rest on the aux slot from a
// second host thread.  Each slot synchronises its own stream between kernels
// while the other's kernels run.  A single batch is not split: two half
// batches repeat the per-batch passes over every user (measured slower at
// 1,000 queries over 1M users, no faster over 100k).
int query_split(rkr_ctx *c, const DataSnap &snap, const float *q, int32_t n, const int32_t *k, int32_t max_k,
                int32_t *ou, int32_t *orank, float *oqip, rkr_query_stats *st, rkr_batch_timing *timing) {
    const int64_t nqb = c->query_batch > 0 ? c->query_batch : 1024;
    const int64_t nb = (n + nqb - 1) / nqb;
    if (c->query_slots < 2 || n < kSplitMinQueries || nb < 2)
        return query_on_slot(c, c->main, snap, q, n, k, max_k, ou, orank, oqip, st, timing);
    if (!c->aux_ready) {
        if (int rc = slot_init(c, c->aux, true, nullptr)) {
            slot_free(c, c->aux);
            return rc;
        }
        c->aux_ready = true;
    }
    const int32_t n1 = (int32_t)std::min<int64_t>(n - 1, (nb + 1) / 2 * nqb);
    const int32_t n2 = n - n1;
    const size_t o = (size_t)n1 * max_k;
    rkr_batch_timing t1{}, t2{};
    int rc2 = RKR_OK;
    const auto t0 = std::chrono::steady_clock::now();
    std::thread th([&] {
        if (hipSetDevice(c->device) != hipSuccess) {
            rc2 = set_err(c, RKR_ERR_HIP, "query: hipSetDevice failed on the second query thread");
            return;
        }
        rc2 = query_on_slot(c, c->aux, snap, q + (size_t)n1 * c->dim, n2, k + n1, max_k, ou + o, orank + o,
                            oqip ? oqip + o : nullptr, st ? st + n1 : nullptr, &t2);
    });
    const int rc1 = query_on_slot(c, c->main, snap, q, n1, k, max_k, ou, orank, oqip, st, &t1);
    th.join();
    if (rc1) return rc1;
    if (rc2) return rc2;
    if (st)
        for (int32_t i = 0; i < n2; ++i) st[n1 + i].query_id += n1;
    if (timing) {
        rkr_batch_timing &t = *timing;
        t = t1;
        t.ip_ms += t2.ip_ms; t.bound_ms += t2.bound_ms; t.prune_ms += t2.prune_ms; t.refine_ms += t2.refine_ms;
        t.recheck_ms += t2.recheck_ms; t.topk_ms += t2.topk_ms; t.h2d_ms += t2.h2d_ms; t.d2h_ms += t2.d2h_ms;
        t.n_batches += t2.n_batches; t.n_refined += t2.n_refined; t.n_rechecked += t2.n_rechecked;
        t.n_screened += t2.n_screened; t.max_screen_err = std::max(t.max_screen_err, t2.max_screen_err);
        t.n_listed += t2.n_listed; t.n_fallback += t2.n_fallback; t.n_coarse_refined += t2.n_coarse_refined;
        t.total_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    }
    return RKR_OK;
}

}  // namespace

extern "C" {

int rkr_query(rkr_ctx *c, const float *queries, int32_t n_query, const int32_t *topk, int32_t max_k,
              int32_t *out_user, int32_t *out_rank, float *out_qip, rkr_query_stats *stats,
              rkr_batch_timing *timing) {
    if (!c) return RKR_ERR_INVALID;
    const DataSnap snap = snap_of(c);
    int rc = validate_queries(c, snap, queries, n_query, topk, max_k);
    if (rc) return rc;
    if (!out_user || !out_rank) return set_err(c, RKR_ERR_INVALID, "query: null output buffer");
    if (timing) std::memset(timing, 0, sizeof(*timing));
    if (n_query == 0) return RKR_OK;
    RKR_HIP(c, hipSetDevice(c->device));
    RKR_HIP(c, hipStreamSynchronize(c->stream));
    if (!c->dedup || n_query < 2)
        return query_split(c, snap, queries, n_query, topk, max_k, out_user, out_rank, out_qip, stats, timing);

    // Identical query vectors (byte-equal) are answered once, with the largest
    // k asked for them: under exact output the answer for k is the first k
    // entries of the answer for any larger k, since (rank, userID) is a total
    // order.  Reference output lists the users its bounds settle first, and that
    // set depends on k (PruneCandidateByBound.hpp:35-77 keeps k-entry heaps), so
    // there only queries equal in vector and k share a run.
    const size_t row = sizeof(float) * (size_t)c->dim;
    const bool by_k = c->output == RKR_OUTPUT_REFERENCE;
    // open addressing over a hash of the row's bytes (and k), byte compare on
    // a hash match: no per-query key copies
    size_t cap = 16;
    while (cap < 2 * (size_t)n_query) cap <<= 1;
    std::vector<int32_t> slot(cap, -1);  // index into reps
    std::vector<int32_t> rep_of((size_t)n_query), reps;
    std::vector<uint64_t> rep_hash;
    for (int32_t i = 0; i < n_query; ++i) {
        const float *qi = queries + (size_t)i * c->dim;
        const uint64_t h = row_hash(qi, row, by_k ? (uint32_t)topk[i] : 0u);
        size_t pos = (size_t)h & (cap - 1);
        int32_t found = -1;
        for (; slot[pos] >= 0; pos = (pos + 1) & (cap - 1)) {
            const int32_t r = slot[pos];
            if (rep_hash[r] == h && std::memcmp(queries + (size_t)reps[r] * c->dim, qi, row) == 0 &&
                (!by_k || topk[reps[r]] == topk[i])) {
                found = r;
                break;
            }
        }
        if (found < 0) {
            found = (int32_t)reps.size();
            slot[pos] = found;
            reps.push_back(i);
            rep_hash.push_back(h);
        }
        rep_of[i] = found;
    }
    const int32_t n_rep = (int32_t)reps.size();
    if (n_rep == n_query)
        return query_split(c, snap, queries, n_query, topk, max_k, out_user, out_rank, out_qip, stats, timing);
    std::vector<float> rq((size_t)n_rep * c->dim);
    std::vector<int32_t> rk((size_t)n_rep, 0);
    for (int32_t j = 0; j < n_rep; ++j) std::memcpy(&rq[(size_t)j * c->dim], queries + (size_t)reps[j] * c->dim, row);
    for (int32_t i = 0; i < n_query; ++i) rk[rep_of[i]] = std::max(rk[rep_of[i]], topk[i]);
    std::vector<int32_t> ru((size_t)n_rep * max_k), rr((size_t)n_rep * max_k);
    std::vector<float> rqip((size_t)n_rep * max_k);
    std::vector<rkr_query_stats> rst(stats ? (size_t)n_rep : 0);
    rc = query_split(c, snap, rq.data(), n_rep, rk.data(), max_k, ru.data(), rr.data(), rqip.data(),
                     stats ? rst.data() : nullptr, timing);
    if (rc) return rc;
    for (int32_t i = 0; i < n_query; ++i) {
        const size_t src = (size_t)rep_of[i] * max_k, dst = (size_t)i * max_k;
        for (int32_t j = 0; j < max_k; ++j) {
            const bool keep = j < topk[i];
            out_user[dst + j] = keep ? ru[src + j] : -1;
            out_rank[dst + j] = keep ? rr[src + j] : -1;
            if (out_qip) out_qip[dst + j] = keep ? rqip[src + j] : -1.0f;
        }
        if (stats) {
            stats[i] = rst[rep_of[i]];
            stats[i].query_id = i;
        }
    }
    return RKR_OK;
}

}  // extern "C"

namespace rkr {

int validate_queries(Ctx *c, const DataSnap &d, const float *queries, int32_t n_query, const int32_t *topk,
                     int32_t max_k) {
    if (!d.table) return set_err(c, RKR_ERR_STATE, "query: no table (build or load one first)");
    if (n_query < 0 || (n_query > 0 && (!queries || !topk)))
        return set_err(c, RKR_ERR_INVALID, "query: null buffer");
    if (max_k <= 0 || max_k > kMaxTopk) return set_err(c, RKR_ERR_INVALID, "query: max_k must be in [1, 4096]");
    for (int32_t i = 0; i < n_query; ++i)
        if (topk[i] <= 0 || topk[i] > max_k || (int64_t)topk[i] > d.n_user)
            return set_err(c, RKR_ERR_INVALID, "query: topk[" + std::to_string(i) + "] = " + std::to_string(topk[i]) +
                                                   " outside [1, min(n_user, max_k)]");
    if (n_query > 0) {
        const double mq = max_abs(queries, (size_t)n_query * c->dim);
        if (mq < 0) return set_err(c, RKR_ERR_INVALID, "query: query vectors must be finite");
        if ((double)c->dim * mq * d.max_abs_user > kScoreLimit)
            return set_err(c, RKR_ERR_INVALID, "query: magnitudes would overflow FP32 scores");
    }
    if (c->output == RKR_OUTPUT_REFERENCE && (d.n_ins > 0 || d.n_del > 0))
        return set_err(c, RKR_ERR_STATE, "query: reference output has no update path; rebuild the table or use exact output");
    return RKR_OK;
}

namespace {

// users per chunk of the coarse histograms and of the list's chunk-major
// order (batches with updates pending): at 1M x 50k (1000 queries) 4096, 8192,
// 16384 and 65536 ran at 258k, 280k, 285k and 279k queries/s (small chunks
// cost histogram workgroups, large ones the exact pass's reuse of user rows
// within a chunk)
constexpr int64_t kCoarseChunk = 16384;
constexpr int32_t kCoarseMinBatch = 8;

// One user of every stride is sampled for the list thresholds: all of up to 16,384
// users (the threshold is then exact), else a sixteenth of them, at least
// 16,384 and at most 65,536.
int64_t sample_stride(int64_t U) {
    const int64_t n = std::min<int64_t>(std::max<int64_t>(U / 16, 16384), 65536);
    return std::max<int64_t>(1, U / n);
}

// List entries of a batch of nq queries: a list is a few hundred users at the
// median and up to a quarter of them for a query that many users rank first
// (longer ones take the full search, as estimated lists past half the entries
// do).  A list entry costs kListBytes with the candidate and refine row it may
// become.
constexpr int64_t kListBytes = 4 * 9;
int64_t list_entries(int64_t U, int64_t nq) {
    const int64_t per = std::min<int64_t>(std::max<int64_t>(U / 64, 4096), 16384);
    return std::min<int64_t>({std::max<int64_t>(nq * per, 2 * std::max<int64_t>(4096, U / 4)), nq * U, INT32_MAX / 2});
}

// How a set of queries is answered: threshold lists (k_list.hip) from matrix-core
// scores of one or three products or from exact scores, or a search over every
// user.  With updates pending the coarse bounds stand for all lists; the plain
// form, and rows too wide for the matrix cores, have lists from exact scores only.
enum Level { kOneProduct, kThreeProducts, kScores, kSearch };  // in the order they are tried
struct Attempt {
    Level level = kOneProduct;
    int64_t entries = 0;          // list entries to make room for, beyond the usual
    const int32_t *rows = nullptr;  // the queries' exact scores are these rows of the slot's scores (ascending)
};
// Fewer users are searched rather than listed from finer scores.
constexpr int64_t kFinerUsers = 16384;
// So are a few queries beside others that are searched: 20 ps a pair.
constexpr int64_t kJoinPairs = 5000000;
// What run_batches left open.
struct Outcome {
    struct Open { int32_t query, thr; };  // and QueryInfo::thr, the reason
    std::vector<Open> open;       // outputs unwritten
    int64_t need = 0;             // pairs of the lists that found no room, as estimated
    int64_t entries = 0;          // list entries there were
    Level level = kSearch;        // what the attempt came to
    bool scores = false;          // the slot holds every query's exact scores, row i the i-th query's
};

// Among many queries, the longest list that is faster than its query's part of a
// search over every user: the search takes 4 ms and 20 us a query at 1M users, a
// listed pair 0.25 ns from matrix-core scores and 0.5 from exact ones, which are
// read twice.  1M users x 1000 queries, 8% of all pairs: 24 ms screened, searched
// 29; 45 plain, searched 31.  (Few long lists are faster all the same, up to a
// quarter of all users: 4 queries, 260k pairs 0.41 ms, searched 4.6.)
int64_t list_share(int64_t U, bool screened) { return std::max<int64_t>(4096, U / (screened ? 12 : 24)); }

// Device batches of query_on_slot.  Queries that the attempt cannot answer (no
// threshold, a list too long or too short) go to out.open.
int run_batches(Ctx *c, Slot &sl, const DataSnap &dv, const float *queries, int32_t n_query, const int32_t *topk,
                int32_t max_k, int32_t *out_user, int32_t *out_rank, float *out_qip, rkr_query_stats *stats,
                rkr_batch_timing &tm, const Attempt &how, Outcome &out) {
    const int64_t U = dv.n_user, I = dv.n_item;
    const int32_t ld = c->ld, d = c->dim;
    const int mode = c->output;
    const bool screened = c->form == RKR_FORM_SCREENED;
    // exact output searches the query table when there is one (exact under
    // the score rule, eps 0); reference output keeps the sampled table
    const bool use_q = mode == RKR_OUTPUT_EXACT && dv.qtable;
    const float *T = use_q ? dv.qtable : dv.table;
    const int32_t *R = use_q ? dv.qranks : dv.ranks;
    const int32_t S = use_q ? dv.n_qs : dv.n_sample;
    const float eps = mode == RKR_OUTPUT_EXACT && !use_q ? dv.table_eps : 0.0f;
    // pending item inserts/deletes: bounds become per-user values (k_update.hip)
    const bool upd = dv.n_ins > 0 || dv.n_del > 0;
    // the QSRP screen (RKR_OPT_QSRP, built by rkr_qsrp_build) replaces the bound
    // stage of exact batches without pending updates
    const bool qsrp = c->qsrp && dv.qsrp_users && mode == RKR_OUTPUT_EXACT && !upd && U > 0;
    const bool listable = !qsrp && how.level != kSearch && c->coarse && mode == RKR_OUTPUT_EXACT && dv.fine.n > 0 && dv.gvals &&
                          dv.guards.n > 0 && U > 0;
    const bool mfma = screened && c->kp > 0 && dv.user_norm;
    const size_t pair_bytes = upd ? 12 : 8;  // <u,q> + buckets, or + two bound values

    // queries per device batch
    int64_t nqb = c->query_batch > 0 ? c->query_batch : 1024;
    {
        const size_t avail = free_bytes(c);
        const int64_t by_mem = (int64_t)(avail / 4 / ((size_t)U * pair_bytes + 1));
        nqb = std::max<int64_t>(1, std::min<int64_t>(nqb, by_mem));
        nqb = std::min<int64_t>(nqb, n_query);
        nqb = std::min<int64_t>(nqb, 65535);
    }
    // The lists, for the screened form and for enough pairs that the search
    // they spare (one user's table row per query, or per batch of 4 and more)
    // outweighs their three launches of about 5 us: at 64k users one plain
    // query is even, and batches of 8 at 4k users.
    const bool list_size = listable && !upd && dv.gcols &&
                           (nqb >= kCoarseMinBatch ? screened || U >= 4096 : U >= (nqb >= 4 ? 8192 : 65536));
    // A list holds k users at least: with a quarter of all users wanted there is
    // nothing to leave out (64 queries, 1000 users, k = 500: 0.33 ms with lists
    // tried first, 0.09 now).
    int64_t k_sum = 0;
    for (int32_t i = 0; i < n_query; ++i) k_sum += topk[i];
    const bool list = list_size && 4 * k_sum <= (int64_t)n_query * U;
    if (list_size && !list && how.level == kOneProduct && how.entries == 0) tm.n_fallback += n_query;
    const bool list_mfma = list && mfma && how.level <= kThreeProducts;
    const int products = how.level == kThreeProducts ? 3 : 1;
    // scores left by the last attempt, of this attempt's queries
    const bool scored = how.rows && !list_mfma && !upd && !qsrp && n_query <= nqb;
    out.level = list_mfma ? how.level : list ? kScores : listable && upd ? kOneProduct : kSearch;
    out.scores = list && !list_mfma && n_query <= nqb;
    // a few users: bounds to candidates in one kernel, its arrays sized for
    // every pair (6 MB at most)
    const bool small = !list && !upd && !qsrp && mode == RKR_OUTPUT_EXACT && U <= kSmallUsers && nqb * U <= (1 << 18);
    // stages are timed by their kernels, or by events where other kernels open them
    const bool use_ev = upd || qsrp;
    // transfers without copy commands
    auto direct_of = [&](const BatchIo &io) { return !use_ev && io.end <= kDirectBytes; };
    int rc;
    const BatchIo io_max(nqb, ld, max_k);
    if ((rc = ensure(c, sl.io, io_max.end, "queries and outputs"))) return rc;
    if ((rc = ensure(c, sl.qip, sizeof(float) * (size_t)nqb * U, "query scores"))) return rc;
    // coarse bucket rows: whole row blocks of 128 users, plus a spare row
    const int64_t ldc = (U + 127) / 128 * 128;
    if (small && (rc = ensure(c, sl.bk, sizeof(uint32_t) * (size_t)(nqb * U), "bucket pairs"))) return rc;
    if (!list && !small && (rc = ensure(c, sl.bk, std::max((pair_bytes - 4) * (size_t)U * nqb, (size_t)ldc * (nqb + 1)),
                              "bucket pairs")))
        return rc;
    if ((rc = ensure(c, sl.hist, sizeof(uint32_t) * hist_words((int32_t)nqb, S), "bound histograms"))) return rc;
    if (qsrp && (rc = ensure(c, sl.q_split, sizeof(float) * (size_t)nqb * (dv.qsrp_ldr + 3), "QSRP query rows")))
        return rc;
    if (small && ((rc = ensure(c, sl.cand, sizeof(int32_t) * 2 * (size_t)(nqb * U), "candidates")) ||
                  (rc = ensure(c, sl.refine_idx, sizeof(int32_t) * 4 * (size_t)(nqb * U), "refine rows"))))
        return rc;
    if (listable && mfma &&
        (rc = ensure(c, sl.q_split, (sizeof(uint16_t) * 2 * c->kp + 2 * sizeof(float)) * (size_t)nqb, "query BF16 rows")))
        return rc;
    // ranks of the searched table's columns (guard placement; the lists and
    // the update path run in exact output only, which searches the query
    // table when there is one)
    const std::vector<int32_t> &hrk = *dv.hrk;
    const GuardCols &gc = dv.guards;
    // an (estimated) list longer than list_max takes the full path instead
    const int64_t list_max = std::max<int64_t>(4096, U / 4);
    int64_t list_cap = 0;
    if (list) {
        // what is held already, or what a quarter of the free budget allows
        const int64_t avail = (int64_t)(free_bytes(c) / 4);
        const int64_t have = std::min<int64_t>({(int64_t)sl.list.bytes / 12, (int64_t)sl.cand.bytes / 8,
                                                (int64_t)sl.refine_idx.bytes / 16, nqb * U, INT32_MAX / 2});
        const int64_t want = std::max(list_entries(U, nqb), std::min<int64_t>({how.entries, nqb * U, INT32_MAX / 2}));
        list_cap = std::max<int64_t>({have, std::min(want, avail / kListBytes), 1});
        out.entries = list_cap;
        if ((rc = ensure(c, sl.list, 12 * (size_t)list_cap, "listed pairs")) ||
            (rc = ensure(c, sl.list_info, sizeof(uint32_t) * (66 * (size_t)nqb + 64), "list thresholds")) ||
            (rc = ensure(c, sl.cand, sizeof(int32_t) * 2 * (size_t)list_cap, "candidates")) ||
            (rc = ensure(c, sl.refine_idx, sizeof(int32_t) * 4 * (size_t)list_cap, "refine rows")))
            return rc;
    }

    // pinned staging: the batch's transfer layout | coarse rows and bin counts
    const size_t stage_io = (io_max.end + 255) & ~(size_t)255;
    if ((rc = ensure_pinned(c, sl.stage, stage_io + std::max<size_t>(sizeof(int32_t) * 12 * (size_t)nqb, 64)))) return rc;
    char *stg = reinterpret_cast<char *>(sl.stage.p);
    int32_t *hcq = reinterpret_cast<int32_t *>(stg + stage_io);
    int32_t *hhc = hcq + 4 * (size_t)nqb;
    if (scored) {  // to the front, where a row is not already (the list of rows on its way through the histograms)
        int32_t first = 0;
        while (first < n_query && how.rows[first] == first) ++first;
        const int32_t n = n_query - first;
        if (n > 0) {
            for (int32_t i = 0; i < n; ++i) hcq[i] = how.rows[first + i] - first;
            RKR_HIP(c, hipMemcpyAsync(sl.hist.p, hcq, sizeof(int32_t) * n, hipMemcpyHostToDevice, sl.stream));
            RKR_HIP(c, launch_keep_rows(sl.stream, reinterpret_cast<float *>(sl.qip.p) + (size_t)first * U, U,
                                        reinterpret_cast<const int32_t *>(sl.hist.p), n));
            RKR_HIP(c, hipStreamSynchronize(sl.stream));  // the staging is the batch's again
        }
    }

    for (int64_t q0 = 0; q0 < n_query; q0 += nqb) {
        const int32_t nq = (int32_t)std::min<int64_t>(nqb, n_query - q0);
        const BatchIo io(nq, ld, max_k);
        const bool direct = direct_of(io);
        char *dev = reinterpret_cast<char *>(sl.io.p);
        float *q_in = reinterpret_cast<float *>(dev);
        QueryInfo *qi = reinterpret_cast<QueryInfo *>(dev + io.info);
        int32_t *q_recheck = reinterpret_cast<int32_t *>(dev + io.recheck);
        ListCounters *ctr = reinterpret_cast<ListCounters *>(dev + io.counters);
        int32_t *o_user = reinterpret_cast<int32_t *>((direct ? stg : dev) + io.out);
        int32_t *o_rank = o_user + (size_t)nq * max_k;
        float *o_qip = reinterpret_cast<float *>(o_rank + (size_t)nq * max_k);
        int32_t *refine_total = &ctr->n_refine;
        uint64_t *const t = use_ev ? nullptr : ctr->t;  // stage stamps
        // few users and queries: the scores' kernel also searches the table
        uint32_t *const small_bk = small && nq <= 16 && eps == 0.0f && !scored ? reinterpret_cast<uint32_t *>(sl.bk.p) : nullptr;
        uint64_t *t_up = reinterpret_cast<uint64_t *>(hcq);  // when the direct upload began
        auto at = [t](int i) { return t ? t + i : nullptr; };
        auto event = [&](int i) { return use_ev ? hipEventRecord(sl.ev[i], sl.stream) : hipSuccess; };
        float *hq = reinterpret_cast<float *>(stg);
        QueryInfo *hqi = reinterpret_cast<QueryInfo *>(stg + io.info);
        const int32_t *h_qrecheck = reinterpret_cast<const int32_t *>(stg + io.recheck);
        const ListCounters *hctr = reinterpret_cast<const ListCounters *>(stg + io.counters);
        const int32_t *ho_user = reinterpret_cast<const int32_t *>(stg + io.out);
        const int32_t *ho_rank = ho_user + (size_t)nq * max_k;
        const float *ho_qip = reinterpret_cast<const float *>(ho_rank + (size_t)nq * max_k);
        float *qip = reinterpret_cast<float *>(sl.qip.p);
        uint32_t *bk = reinterpret_cast<uint32_t *>(sl.bk.p);

        // largest |query value| of the batch (validated finite)
        const double q_amax = max_abs(queries + (size_t)q0 * d, (size_t)nq * d);
        for (int32_t i = 0; i < nq; ++i) {
            float *dst = &hq[(size_t)i * ld];
            std::memcpy(dst, queries + (size_t)(q0 + i) * d, sizeof(float) * d);
            for (int32_t k = d; k < ld; ++k) dst[k] = 0.0f;
            hqi[i] = QueryInfo{};
            hqi[i].topk = topk[q0 + i];
        }
        std::memset(stg + io.recheck, 0, io.out - io.recheck);
        const bool plain_list = list && !list_mfma;  // its sample histogram is cleared here
        if (direct) {
            RKR_HIP(c, launch_upload(sl.stream, stg, dev, io.out, plain_list ? sl.list_info.p : nullptr,
                                     plain_list ? sizeof(uint32_t) * 64 * (size_t)nq : 0, t_up));
        } else {
            RKR_HIP(c, hipEventRecord(sl.ev[0], sl.stream));
            RKR_HIP(c, hipMemcpyAsync(dev, stg, io.out, hipMemcpyHostToDevice, sl.stream));
            RKR_HIP(c, hipEventRecord(sl.ev[1], sl.stream));
        }
        int32_t *lbv = reinterpret_cast<int32_t *>(bk);
        int32_t *ubv = lbv + (size_t)nq * U;
        const int64_t cu = chunk_users(U, nq, c->n_cu);
        uint32_t *ghist = reinterpret_cast<uint32_t *>(sl.hist.p);
        // a few queries with updates pending are answered faster by the full
        // path: the coarse kernel converts every user row once per launch
        const bool coarse = listable && upd && mfma && nq >= kCoarseMinBatch;
        uint16_t *q_hi = reinterpret_cast<uint16_t *>(sl.q_split.p);
        uint16_t *q_lo = q_hi + (size_t)nqb * c->kp;
        float *qn = reinterpret_cast<float *>(q_lo + (size_t)nqb * c->kp);
        float *qcs = qn + nqb;  // error scales of the one-product estimate
        // e = C ||u|| cs + floor, C = 1 + 2^-20 covering the FP32 evaluation of
        // that product and sum
        const float est_C = 1.0f + 0x1p-20f;
        const float est_floor = std::nextafter(
            (float)(((double)screen_abs_floor(c->kp, dv.max_abs_user, q_amax) + (double)eps) * (1.0 + std::ldexp(1.0, -18))),
            INFINITY);
        ListLaunch LL{};
        uint32_t *bk_c = nullptr;
        std::vector<int32_t> deep_check;  // update path: queries listed without the deepest bin
        if (list) {
            LL.n_user = U; LL.nq = nq; LL.S = S; LL.Kp = c->kp; LL.n_cu = c->n_cu;
            LL.user_hi = dv.user_hi; LL.user_norm = dv.user_norm; LL.gvals = dv.gvals; LL.gcols = dv.gcols; LL.pitch = dv.gpitch;
            LL.q_hi = q_hi; LL.q_cs = products == 1 ? qcs : qn; LL.C = products == 1 ? est_C : c->screen_C;
            LL.fc = dv.fine; LL.floor = est_floor; LL.eps = eps;
            LL.qip = qip; LL.stride = sample_stride(U); LL.cap = list_max; LL.share = list_share(U, list_mfma); LL.list_cap = list_cap;
            // An estimate is off by what the sample is; without the pairs that the
            // scores' error adds it would be half of what comes.
            LL.room = list_cap >= (int64_t)nq * U ? list_cap : list_mfma ? list_cap / 4 * 3 : list_cap / 2;
            // A list that one product's error makes longer than this is cheaper
            // from three (1.3 us a query at 1M users, 0.25 ns a pair).
            LL.band = list_mfma && products == 1 && U >= kFinerUsers ? std::max<int64_t>(4096, U / 64) : U;
            LL.products = products;
            LL.user_lo = dv.user_lo; LL.q_lo = q_lo;
            LL.hist = reinterpret_cast<uint32_t *>(sl.list_info.p);
            LL.order = reinterpret_cast<int32_t *>(LL.hist + 64 * (size_t)nq);
            LL.colg = LL.order + nq;
            LL.qi = qi; LL.ctr = ctr; LL.t_bound = at(kTimeBound); LL.t_prune = at(kTimePrune);
            LL.cl_u = reinterpret_cast<int32_t *>(sl.list.p);
            LL.cl_b = LL.cl_u + list_cap;
            LL.raw_u = LL.cl_u;
            LL.raw_b = LL.cl_b;
            if (nq > kFilterQueries) {  // as listed: where the candidates go later
                LL.raw_u = reinterpret_cast<int32_t *>(sl.cand.p);
                LL.raw_b = LL.raw_u + list_cap;
                LL.g_cnt = ghist;
                LL.g_cur = LL.g_cnt + nq;
                LL.g_off = LL.g_cur + nq;
            }
            bk_c = reinterpret_cast<uint32_t *>(LL.cl_b + list_cap);
        }
        if (list_mfma) {
            RKR_HIP(c, launch_prep_items(sl.stream, q_in, nq, ld, d, c->kp, q_hi, q_lo, qn, qcs, dv.rho, c->coarse_g1,
                                         c->coarse_grule, LL.hist, at(kTimeIp)));
            RKR_HIP(c, launch_list_screen(sl.stream, LL));
            RKR_HIP(c, event(2));
            RKR_HIP(c, launch_list_exact(sl.stream, LL, dv.users, q_in, ld, d, T, false, bk_c));
            RKR_HIP(c, event(3));
        } else if (coarse) {
            // coarse buckets on the matrix cores, the coarse k-th bound and
            // list sizes; exact scores and bound values of the listed users
            RKR_HIP(c, launch_prep_items(sl.stream, q_in, nq, ld, d, c->kp, q_hi, q_lo, qn, qcs, dv.rho, c->coarse_g1,
                                         c->coarse_grule));
            uint8_t *cb = reinterpret_cast<uint8_t *>(bk);
            CoarseLaunch L{};
            L.user_norm = dv.user_norm; L.gvals = dv.gvals; L.user_hi = dv.user_hi; L.n_user = U; L.gc = gc;
            L.q_hi = q_hi; L.q_cs = qcs; L.nq = nq; L.Kp = c->kp; L.C = est_C; L.abs_floor = est_floor; L.cb = cb;
            L.ldc = ldc; L.spare_row = nqb;
            L.grid_cap = (int64_t)c->n_cu * coarse_first_pass_wgs(c->kp / 32);
            RKR_HIP(c, launch_ip_coarse(sl.stream, L));
            RKR_HIP(c, event(2));
            // coarse chunks: a fixed user count, so launches over few queries
            // still fill the device and the list stays chunk-major
            const int64_t ccu = kCoarseChunk;
            const int64_t n_chunk = (U + ccu - 1) / ccu;
            // part | cq | loc | ctot | cbase | hcnt
            if ((rc = ensure(c, sl.list_info, sizeof(uint32_t) * (17 * (size_t)nq * n_chunk + 12 * (size_t)nqb +
                                                                  2 * (size_t)n_chunk + 64),
                             "coarse counts")))
                return rc;
            uint32_t *part = reinterpret_cast<uint32_t *>(sl.list_info.p);
            int32_t *cq = reinterpret_cast<int32_t *>(part + 16 * (size_t)nq * n_chunk);
            int32_t *loc = cq + 4 * (size_t)nqb;
            int32_t *ctot = loc + (size_t)nq * n_chunk;
            int32_t *cbase = ctot + n_chunk;
            int32_t *hcnt = cbase + n_chunk;
            RKR_HIP(c, launch_coarse_kth(sl.stream, cb, ldc, U, nq, ccu, gc.n, part, qi, cq, hcnt));
            RKR_HIP(c, hipMemcpyAsync(hcq, cq, sizeof(int32_t) * 4 * nq, hipMemcpyDeviceToHost, sl.stream));
            RKR_HIP(c, hipMemcpyAsync(hhc, hcnt, sizeof(int32_t) * 8 * nq, hipMemcpyDeviceToHost, sl.stream));
            RKR_HIP(c, hipStreamSynchronize(sl.stream));
            int64_t n_listed = 0;
            for (int32_t i = 0; i < nq; ++i) {
                int32_t *e = &hcq[(size_t)i * 4];
                if (e[0] >= 0) {
                    // pending inserts move ranks: a user at or above guard m has
                    // rank <= R[j_m] + ins_gmax[m], so the k-th bound is at most
                    // V = R[j_beta] + ins_gmax[beta]; a user below guard c_hi - 1
                    // has rank >= R[j_{c_hi - 1}] + 1 - n_del, and is listed when
                    // that can be <= V
                    const int64_t V = (int64_t)hrk[gc.col[e[0]]] + dv.ins_gmax[e[0]];
                    int32_t bl = 0;
                    while (bl < gc.n && (int64_t)hrk[gc.col[bl]] + 1 - dv.n_del <= V) ++bl;
                    if (bl >= gc.n) {
                        // users below the deepest guard are left out; the
                        // exact k-th value then has to stay below their
                        // lowest possible rank (checked after the selection)
                        bl = gc.n - 1;
                        deep_check.push_back(i);
                    }
                    int64_t n = 0;
                    for (int32_t cc = 0; cc <= bl; ++cc) n += hhc[(size_t)i * 8 + cc];
                    e[0] = bl;
                    e[1] = (int32_t)std::min<int64_t>(n, INT32_MAX);
                }
                if (e[0] < 0 || e[1] > list_max) {
                    out.open.push_back({(int32_t)(q0 + i), kNoList});
                    e[0] = -1;
                    e[1] = 0;
                }
                e[2] = (int32_t)n_listed;
                e[3] = 0;
                n_listed += e[1];
            }
            tm.n_listed += n_listed;
            if (n_listed >= INT32_MAX) return set_err(c, RKR_ERR_NOMEM, "query: coarse list exceeds 2^31; lower the query batch");
            if ((rc = ensure(c, sl.list, 8 * (size_t)std::max<int64_t>(n_listed, 1), "coarse list"))) return rc;
            int32_t *cl_u = reinterpret_cast<int32_t *>(sl.list.p);
            int32_t *cl_b = cl_u + std::max<int64_t>(n_listed, 1);
            RKR_HIP(c, hipMemcpyAsync(cq, hcq, sizeof(int32_t) * 4 * nq, hipMemcpyHostToDevice, sl.stream));
            RKR_HIP(c, launch_coarse_compact(sl.stream, cb, ldc, U, nq, ccu, part, cq, loc, ctot, cbase, cl_u, cl_b));
            // bound values of the listed pairs only (the rest are ruled
            // out), then the value selection of the update path; the
            // bound arrays reuse the coarse rows, read by now
            RKR_HIP(c, hipMemsetD32Async(reinterpret_cast<hipDeviceptr_t>(lbv), kNoBound, 2 * (size_t)nq * U, sl.stream));
            RKR_HIP(c, launch_coarse_exact_upd(sl.stream, dv.users, q_in, ld, d, T, S, R, dv.n_item_base, eps, gc, cl_u,
                                               cl_b, n_listed, dv.side_ins, dv.n_ins, dv.ld_ins, dv.side_del, dv.n_del,
                                               dv.ld_del, U, lbv, ubv, qip));
            RKR_HIP(c, launch_kth_values(sl.stream, lbv, ubv, U, nq, cu, ghist, qi));
            RKR_HIP(c, event(3));
        } else if (qsrp) {
            // QSRP screen: rotated queries and their part norms, the left-part
            // scores over the first check_dim dimensions, bounds from the
            // partial-dimension interval and the regression, the k-th bound
            // over those, then the exact score and table search for the users
            // they keep, and the k-th bound again (the exact path's from here)
            float *qrot = reinterpret_cast<float *>(sl.q_split.p);
            float *qpn = qrot + (size_t)nqb * dv.qsrp_ldr;
            RKR_HIP(c, launch_scores_store(sl.stream, q_in, nq, ld, dv.qsrp_rot, d, ld, d, qrot,
                                           dv.qsrp_ldr, true));
            RKR_HIP(c, launch_qsrp_qnorms(sl.stream, qrot, dv.qsrp_ldr, q_in, ld, d, dv.qsrp_cd, nq, qpn));
            RKR_HIP(c, launch_scores_store(sl.stream, dv.qsrp_users, U, dv.qsrp_ldr, qrot, nq, dv.qsrp_ldr,
                                           dv.qsrp_cd, qip, U, false));
            RKR_HIP(c, event(2));
            // eps widens the interval as the exact path widens its search; the
            // floor covers gradual underflow in the d products of a score
            const float absf = std::nextafter((float)((double)eps + (double)d * std::ldexp(1.0, -140)), INFINITY);
            RKR_HIP(c, launch_qsrp_bounds(sl.stream, qip, U, nq, dv.qsrp_par, qpn, dv.qsrp_gcd, dv.qsrp_crot, absf,
                                          dv.n_sample, use_q ? dv.qcol : nullptr, S, bk));
            RKR_HIP(c, launch_hist_kth(sl.stream, bk, U, S, R, I, nq, mode, 0, cu, ghist, qi));
            RKR_HIP(c, launch_qsrp_exact(sl.stream, dv.users, q_in, ld, d, T, S, eps, U, nq, qi, qip, bk));
            RKR_HIP(c, event(3));
            RKR_HIP(c, launch_hist_kth(sl.stream, bk, U, S, R, I, nq, mode, 0, cu, ghist, qi));
        } else {
            // <u, q> for every (query, user): qip[b * U + u]
            if (!scored && nq <= 16)
                RKR_HIP(c, launch_gemv_panels(sl.stream, dv.usersT, U, ld, d, q_in, nq, qip, T, S, small_bk, at(kTimeIp)));
            else if (!scored) RKR_HIP(c, launch_scores_store(sl.stream, dv.users, U, ld, q_in, nq, ld, d, qip, U, false, at(kTimeIp)));
            RKR_HIP(c, event(2));
            if (list) {
                if (!direct) RKR_HIP(c, hipMemsetAsync(LL.hist, 0, sizeof(uint32_t) * 64 * (size_t)nq, sl.stream));
                RKR_HIP(c, launch_list_scores(sl.stream, LL));
                RKR_HIP(c, launch_list_exact(sl.stream, LL, dv.users, q_in, ld, d, T, true, bk_c));
                RKR_HIP(c, event(3));
            } else if (upd) {
                RKR_HIP(c, launch_bounds_upd(sl.stream, qip, T, dv.gvals, dv.fine, U, S, R, dv.n_item_base, eps, dv.side_ins,
                                             dv.n_ins, dv.ld_ins, dv.side_del, dv.n_del, dv.ld_del, nq, lbv, ubv));
                RKR_HIP(c, event(3));
                RKR_HIP(c, launch_kth_values(sl.stream, lbv, ubv, U, nq, cu, ghist, qi));
            } else if (!small) {
                RKR_HIP(c, launch_bounds(sl.stream, qip, T, U, S, nq, eps, mode == RKR_OUTPUT_REFERENCE ? 1 : 0, bk,
                                         at(kTimeBound)));
                RKR_HIP(c, event(3));
                RKR_HIP(c, launch_hist_kth(sl.stream, bk, U, S, R, I, nq, mode,
                                           (mode == RKR_OUTPUT_EXACT && eps == 0.0f) ? 1 : 0, cu, ghist, qi, at(kTimePrune)));
            }
        }
        // With lists every candidate is a listed pair, so the list's entries
        // bound the candidate and refine arrays and the batch goes on without
        // waiting for the counts (the refinement and top-k read them on the
        // device).  Otherwise the counts size them.
        int64_t total = small ? nqb * U : list_cap, total_cand = total;
        if (!list && !small) {
            RKR_HIP(c, launch_offsets(sl.stream, qi, nq, refine_total));
            RKR_HIP(c, hipMemcpyAsync(hqi, qi, sizeof(QueryInfo) * nq, hipMemcpyDeviceToHost, sl.stream));
            RKR_HIP(c, hipStreamSynchronize(sl.stream));
            // (the device's offsets are 32-bit sums: past that the check below is on these)
            total = total_cand = 0;
            for (int32_t i = 0; i < nq; ++i) {
                total += (int64_t)hqi[i].n_settled + hqi[i].n_cand;
                total_cand += hqi[i].n_cand;
            }
        }
        if (!deep_check.empty()) {
            // a user below the deepest guard has rank >= r[j_last] + 1 - n_del:
            // the selection over the listed users is exact when the k-th value
            // L (QueryInfo.gamma of the value selection) is below that
            const int64_t floor_rank = (int64_t)hrk[gc.col[gc.n - 1]] + 1 - dv.n_del;
            for (int32_t i : deep_check)
                if (hcq[(size_t)i * 4] >= 0 && (int64_t)hqi[i].gamma >= floor_rank)
                    out.open.push_back({(int32_t)(q0 + i), kNoList});
        }
        if (total >= INT32_MAX) return set_err(c, RKR_ERR_NOMEM, "query: candidate count exceeds 2^31; lower the query batch");
        const size_t cap = (size_t)std::max<int64_t>(total, 1);
        const size_t rcap = (size_t)std::max<int64_t>(total_cand, 1);
        if ((rc = ensure(c, sl.cand, sizeof(int32_t) * 2 * cap, "candidates"))) return rc;
        if ((rc = ensure(c, sl.refine_idx, sizeof(int32_t) * 4 * rcap, "refine rows"))) return rc;
        int32_t *cand_user = reinterpret_cast<int32_t *>(sl.cand.p);
        int32_t *cand_rank = cand_user + cap;
        int32_t *refine_user = reinterpret_cast<int32_t *>(sl.refine_idx.p);
        int32_t *refine_query = refine_user + rcap;
        float *refine_thr = reinterpret_cast<float *>(refine_query + rcap);
        int32_t *cnt = reinterpret_cast<int32_t *>(refine_thr + rcap);

        if (small)
            RKR_HIP(c, launch_small_select(sl.stream, qip, T, small_bk, U, S, R, I, nq, eps, qi, ctr, cand_user, cand_rank,
                                           refine_user, refine_query, refine_thr, cnt));
        else if (list)
            RKR_HIP(c, launch_list_final(sl.stream, LL, bk_c, R, I, cand_user, cand_rank, refine_user, refine_query,
                                         refine_thr, cnt));
        else if (upd)
            RKR_HIP(c, launch_compact_values(sl.stream, lbv, ubv, qip, U, nq, cu, qi, cand_user, cand_rank,
                                             refine_total, refine_user, refine_query, refine_thr, cnt));
        else
            RKR_HIP(c, launch_compact(sl.stream, bk, qip, U, S, R, I, nq, mode, cu, qi, cand_user, cand_rank,
                                      refine_total, refine_user, refine_query, refine_thr, cnt));
        // without a list the rows' bound is the candidates' count; a list over a
        // table with every top rank leaves few rows, whatever its capacity
        const bool many = !list || !use_q;
        // refinement + top-k; re-run when the recheck list overflowed
        for (int attempt = 0; attempt < 3; ++attempt) {
            int64_t rec_cap = 0;
            if (screened) {
                const int64_t want = std::max<int64_t>(1 << 20, (int64_t)sl.recheck.bytes / 16);
                if ((rc = ensure(c, sl.recheck, 16 * (size_t)want, "recheck list"))) return rc;
                rec_cap = (int64_t)(sl.recheck.bytes / 16);
            }
            if (attempt > 0) {  // the compaction cleared the counts, the upload the recheck counters
                RKR_HIP(c, hipMemsetAsync(cnt, 0, sizeof(int32_t) * rcap, sl.stream));
                RKR_HIP(c, hipMemsetAsync(q_recheck, 0, sizeof(int32_t) * (size_t)nq, sl.stream));
                RKR_HIP(c, hipMemsetAsync(&ctr->n_recheck, 0, sizeof(int32_t) * 2, sl.stream));
            }
            RKR_HIP(c, event(4));
            // events 4..8, or the stamps, bracket exactly the refinement (or screening) kernel
            if (screened) {
                ScreenLaunch L{};
                L.users = dv.users; L.user_norm = dv.user_norm;
                L.user_hi = dv.user_hi; L.user_lo = dv.user_lo;
                L.item_hi = dv.item_hi; L.item_lo = dv.item_lo; L.item_norm = dv.item_norm;
                L.n_item = I; L.ld = ld; L.K = d; L.Kp = c->kp;
                L.rows_user = refine_user; L.rows_thr = refine_thr; L.n_rows_dev = refine_total;
                L.max_rows = (int64_t)rcap; L.C = c->screen_C; L.abs_floor = dv.screen_abs;
                L.cnt = cnt; L.recheck_n = &ctr->n_recheck; L.recheck = sl.recheck.p; L.recheck_cap = rec_cap;
                L.n_cu = c->n_cu;
                L.chunk_items = c->screen_chunk > 0 ? c->screen_chunk : (1 << 30);
                L.t = at(kTimeRefine);
                L.rows_per_wave = c->screen_rows > 0 ? c->screen_rows : 32;
                RKR_HIP(c, launch_refine_screen(sl.stream, L));
                RKR_HIP(c, event(8));
                RKR_HIP(c, launch_recheck(sl.stream, dv.users, dv.items, ld, d, refine_user, refine_thr, refine_query,
                                          &ctr->n_recheck, sl.recheck.p, rec_cap, cnt, q_recheck, &ctr->max_err_bits,
                                          at(kTimeRecheck)));
            } else {
                RKR_HIP(c, launch_refine_count(sl.stream, dv.users, dv.items, I, ld, d, refine_user, refine_thr,
                                               refine_total, (int64_t)rcap, cnt, many, at(kTimeRefine)));
                RKR_HIP(c, event(8));
            }
            RKR_HIP(c, event(5));
            RKR_HIP(c, launch_topk(sl.stream, qi, nq, cand_user, cand_rank, cnt, qip, U, max_k, o_user, o_rank, o_qip, at(kTimeTopk),
                                   at(kTimeEnd),
                                   direct ? HostResult{hqi, reinterpret_cast<int32_t *>(stg + io.recheck),
                                                       reinterpret_cast<ListCounters *>(stg + io.counters), q_recheck, ctr}
                                          : HostResult{}));
            RKR_HIP(c, event(6));
            if (!direct) {
                // query info, counters and outputs in one copy (the device layout)
                RKR_HIP(c, hipMemcpyAsync(stg + io.info, dev + io.info, io.end - io.info, hipMemcpyDeviceToHost, sl.stream));
                RKR_HIP(c, hipEventRecord(sl.ev[7], sl.stream));
            }
            RKR_HIP(c, hipStreamSynchronize(sl.stream));
            const int64_t n_recheck = hctr->n_recheck;
            if (!screened || n_recheck <= rec_cap) break;
            // the list overflowed: grow it and run the refinement again
            const size_t need = 16 * ((size_t)n_recheck + (size_t)n_recheck / 4 + 1024);
            dev_free(c, sl.recheck.p, sl.recheck.bytes);
            sl.recheck.p = nullptr;
            sl.recheck.bytes = 0;
            if ((rc = ensure(c, sl.recheck, need, "recheck list"))) return rc;
            if (attempt == 2) return set_err(c, RKR_ERR_NOMEM, "query: recheck list kept overflowing");
        }
        if (list) {
            for (int32_t i = 0; i < nq; ++i)
                if (hqi[i].thr < 0) out.open.push_back({(int32_t)(q0 + i), hqi[i].thr});
            out.need += (int64_t)hctr->n_need;
            if ((int64_t)hctr->n_list <= list_cap) tm.n_listed += (int64_t)hctr->n_list;  // else no stage read the list
            tm.n_coarse_refined += hctr->n_finer;
        }
        if (qsrp)
            for (int32_t i = 0; i < nq; ++i) tm.n_listed += hqi[i].n_screen;

        std::memcpy(out_user + (size_t)q0 * max_k, ho_user, sizeof(int32_t) * (size_t)nq * max_k);
        std::memcpy(out_rank + (size_t)q0 * max_k, ho_rank, sizeof(int32_t) * (size_t)nq * max_k);
        if (out_qip) std::memcpy(out_qip + (size_t)q0 * max_k, ho_qip, sizeof(float) * (size_t)nq * max_k);
        if (stats) {
            for (int32_t i = 0; i < nq; ++i) {
                rkr_query_stats &st = stats[q0 + i];
                std::memset(&st, 0, sizeof(st));
                st.query_id = (int32_t)(q0 + i);
                st.n_candidate = hqi[i].n_cand;
                st.n_refine_user = hqi[i].n_refine;
                if (mode == RKR_OUTPUT_EXACT) {
                    st.n_result_user = hqi[i].n_cand - hqi[i].n_refine;
                    st.n_prune_user = (int32_t)(U - hqi[i].n_cand);
                } else {
                    st.n_result_user = hqi[i].n_settled;
                    st.n_prune_user = (int32_t)(U - hqi[i].n_settled - hqi[i].n_cand);
                }
                // inner products: every user's (QSRP: the screen's survivors), then the refinement's
                st.ip_cost = (qsrp ? (int64_t)hqi[i].n_screen : U) + (int64_t)hqi[i].n_refine * I;
                if (screened) {
                    st.n_screened = (int64_t)hqi[i].n_refine * I;
                    st.n_rechecked = h_qrecheck[i];
                }
            }
        }
        if (!direct) tm.h2d_ms += ev_ms(sl.ev, 0, 1);
        if (use_ev) {
            tm.ip_ms += ev_ms(sl.ev, 1, 2);
            tm.bound_ms += ev_ms(sl.ev, 2, 3);
            tm.prune_ms += ev_ms(sl.ev, 3, 4);
            tm.refine_ms += ev_ms(sl.ev, 4, 8);
            tm.recheck_ms += ev_ms(sl.ev, 8, 5);
            tm.topk_ms += ev_ms(sl.ev, 5, 6);
            tm.d2h_ms += ev_ms(sl.ev, 6, 7);
        } else {
            // a stage without a kernel of its own starts with the next
            uint64_t ts[kTimeEnd + 1];
            for (int i = 0; i <= kTimeEnd; ++i) ts[i] = hctr->t[i];
            if (direct) {  // the last workgroup's end, from the low words
                // (a query without candidates can be done before the first workgroup stamps the start)
                int32_t end = 0;
                for (int32_t i = 0; i < nq; ++i) end = std::max(end, (int32_t)((uint32_t)hqi[i].pad - (uint32_t)ts[kTimeTopk]));
                ts[kTimeEnd] = ts[kTimeTopk] + (uint32_t)end;
            }
            for (int i = kTimeEnd - 1; i >= 0; --i)
                if (ts[i] == 0) ts[i] = ts[i + 1];
            auto ms = [&](int i) { return ts[i + 1] > ts[i] ? (double)(ts[i + 1] - ts[i]) / c->clock_khz : 0.0; };
            tm.ip_ms += ms(kTimeIp);
            tm.bound_ms += ms(kTimeBound);
            tm.prune_ms += ms(kTimePrune);
            tm.refine_ms += ms(kTimeRefine);
            tm.recheck_ms += ms(kTimeRecheck);
            tm.topk_ms += ms(kTimeTopk);
            if (direct) {  // the outputs leave within the top-k
                tm.h2d_ms += ts[kTimeIp] > *t_up ? (double)(ts[kTimeIp] - *t_up) / c->clock_khz : 0.0;
            } else {  // what is left of the time after the upload
                const double kernels = ts[kTimeEnd] > ts[kTimeIp] ? (double)(ts[kTimeEnd] - ts[kTimeIp]) / c->clock_khz : 0.0;
                tm.d2h_ms += std::max(0.0, ev_ms(sl.ev, 1, 7) - kernels);
            }
        }
        tm.n_batches += 1;
        tm.n_refined += hctr->n_refine;
        if (screened) {
            tm.n_rechecked += hctr->n_recheck;
            tm.n_screened += (int64_t)hctr->n_refine * I;
            float e;
            std::memcpy(&e, &hctr->max_err_bits, sizeof(e));
            tm.max_screen_err = std::max(tm.max_screen_err, (double)e);
        }
    }
    return RKR_OK;
}

}  // namespace

namespace {

// Queries that wait for an attempt.
struct Group {
    Attempt how;
    std::vector<int32_t> idx;  // ascending
};

// Answers n queries: every attempt's open queries join the group of their next
// one -- lists that only found no room once more with more of it, the others
// finer scores or the search -- and the groups are taken in the order of their
// levels, so that the search runs once.
int answer(Ctx *c, Slot &sl, const DataSnap &dv, const float *queries, int32_t n, const int32_t *topk, int32_t max_k,
           int32_t *out_user, int32_t *out_rank, float *out_qip, rkr_query_stats *stats, rkr_batch_timing &tm) {
    Outcome o;
    int rc = run_batches(c, sl, dv, queries, n, topk, max_k, out_user, out_rank, out_qip, stats, tm, Attempt{}, o);
    if (rc || o.open.empty()) return rc;
    const int32_t d = c->dim;
    const bool upd = dv.n_ins > 0 || dv.n_del > 0;
    std::vector<Group> todo;
    std::vector<int32_t> scored;  // queries whose scores the slot holds, row by row
    auto put = [&](Level level, int64_t entries, int32_t q) {
        for (Group &g : todo)
            if (g.how.level == level && (g.how.entries > 0) == (entries > 0)) {
                g.how.entries = std::max(g.how.entries, entries);
                g.idx.push_back(q);
                return;
            }
        todo.emplace_back();
        todo.back().how.level = level;
        todo.back().how.entries = entries;
        todo.back().idx.push_back(q);
    };
    // the open queries of an attempt on `idx` (null: all queries in order)
    auto sort_out = [&](const Attempt &how, const std::vector<int32_t> *idx, int32_t m) {
        int64_t n_room = 0, n_search = 0;
        for (const auto &x : o.open) {
            n_room += x.thr == kNoRoom;
            n_search += x.thr == kNoList;
        }
        // an attempt of their own (100 us) costs these more than joining the others' search
        const bool join = n_search > 0 && ((int64_t)o.open.size() - n_search) * dv.n_user < kJoinPairs;
        const int64_t entries = std::max<int64_t>(1, 2 * (o.need + o.need / 8));
        const bool again = how.entries == 0 && n_room > 0 && (n_room < m || entries > o.entries);
        const Level finer = upd || o.level == kScores || dv.n_user < kFinerUsers ? kSearch
                            : o.level == kOneProduct                            ? kThreeProducts
                                                                                : kScores;
        for (const auto &x : o.open) {
            const int32_t q = idx ? (*idx)[x.query] : x.query;
            if (join) put(kSearch, 0, q);
            else if (again && x.thr == kNoRoom) put(o.level, entries, q);
            else put(x.thr == kNoList ? kSearch : finer, 0, q);
        }
        scored.clear();
        if (o.scores)
            for (int32_t i = 0; i < m; ++i) scored.push_back(idx ? (*idx)[i] : i);
    };
    sort_out(Attempt{}, nullptr, n);
    while (!todo.empty()) {
        const auto first = std::min_element(todo.begin(), todo.end(), [](const Group &x, const Group &y) {
            return x.how.level != y.how.level ? x.how.level < y.how.level : x.how.entries < y.how.entries;
        });
        Group g = std::move(*first);
        todo.erase(first);
        std::sort(g.idx.begin(), g.idx.end());
        const int32_t m = (int32_t)g.idx.size();
        // the scores of the last attempt, if it held them all
        std::vector<int32_t> rows;
        if (g.how.level >= kScores)
            for (size_t i = 0; i < scored.size() && rows.size() < g.idx.size(); ++i)
                if (scored[i] == g.idx[rows.size()]) rows.push_back((int32_t)i);
        if (rows.size() == g.idx.size()) g.how.rows = rows.data();
        std::vector<float> q((size_t)m * d), qip((size_t)m * max_k);
        std::vector<int32_t> k((size_t)m), u((size_t)m * max_k), r((size_t)m * max_k);
        std::vector<rkr_query_stats> st(stats ? (size_t)m : 0);
        for (int32_t i = 0; i < m; ++i) {
            std::memcpy(&q[(size_t)i * d], queries + (size_t)g.idx[i] * d, sizeof(float) * d);
            k[i] = topk[g.idx[i]];
        }
        o = Outcome{};
        rc = run_batches(c, sl, dv, q.data(), m, k.data(), max_k, u.data(), r.data(), qip.data(), stats ? st.data() : nullptr,
                         tm, g.how, o);
        if (rc) return rc;
        if (o.level == kSearch) tm.n_fallback += m;
        // rows of a query that is still open are written again
        for (int32_t i = 0; i < m; ++i) {
            const size_t to = (size_t)g.idx[i] * max_k, from = (size_t)i * max_k;
            std::memcpy(out_user + to, &u[from], sizeof(int32_t) * max_k);
            std::memcpy(out_rank + to, &r[from], sizeof(int32_t) * max_k);
            if (out_qip) std::memcpy(out_qip + to, &qip[from], sizeof(float) * max_k);
            if (stats) {
                stats[g.idx[i]] = st[i];
                stats[g.idx[i]].query_id = g.idx[i];
            }
        }
        sort_out(g.how, &g.idx, m);
    }
    return RKR_OK;
}

}  // namespace

int query_on_slot(Ctx *c, Slot &sl, const DataSnap &dv, const float *queries, int32_t n_query, const int32_t *topk,
                  int32_t max_k, int32_t *out_user, int32_t *out_rank, float *out_qip, rkr_query_stats *stats,
                  rkr_batch_timing *timing) {
    using clock = std::chrono::steady_clock;
    const auto t_start = clock::now();
    rkr_batch_timing tm{};
    const int rc = answer(c, sl, dv, queries, n_query, topk, max_k, out_user, out_rank, out_qip, stats, tm);
    if (rc) return rc;
    tm.total_ms = std::chrono::duration<double, std::milli>(clock::now() - t_start).count();
    if (timing) *timing = tm;
    return RKR_OK;
}

}  // namespace rkr
