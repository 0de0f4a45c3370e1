/*
 * stc_query.hip — batched queries over the resident state.
 *
 * Object-history, square-range and pair queries (semantics at stc_query_batch in
 * include/stcdb.h) are answered from three sources in one pass each:
 *   - the live meetings: a grid-stride scan over their ids, boxes or both, live
 *     ones (end == last step) matched in both directions;
 *   - the memtable records: one thread per record;
 *   - the runs kept in HBM: object and pair queries look the object's CTF up
 *     through the run's sids and search its packed keys (a wave each, 64 probes
 *     a round), which a CTF stores sorted by pid (as CTF::search_SSTable does,
 *     step_merge.cpp:528);
 *     range queries scan the CTFs whose decoded boxes can reach the query box
 *     (one block per query and CTF) and the oversize buffer.
 * Object and pair queries are found per meeting through a small open-addressed
 * hash of the queried ids; range queries through a 64 x 64 grid of the map,
 * each (meeting, query) pair reported from the grid cell that holds the low
 * corner of their intersection, so exactly once.
 */
#include "stc_query.h"

#include <algorithm>
#include <cmath>
#include <cstring>

#define QGRID 64
#define QFINE 256 /* cells a side of the scans' range filter */
#define QSTAGE 48 /* hits a wave gathers before it reserves room for them */
#define QLDS 4096 /* batches up to this many queries count in LDS, block by block */
#define MASK26 ((1u << 26) - 1u)

struct QDev {
    const stc_query *q;
    const uint32_t *oh_key;          /* queried ids, 0xFFFFFFFF = empty slot */
    const int32_t *oh_head;          /* first query of the id */
    const int32_t *q_next;           /* next query with the same id, -1 ends */
    uint32_t oh_bits;                /* 0: no object or pair queries */
    uint32_t n_range;
    const uint32_t *g_start;         /* [QGRID * QGRID + 1] range queries by grid cell */
    const uint32_t *g_list;
    const uint32_t *filter;          /* [2^f_bits / 32] a bit per hash of a queried id, then [QGRID * QGRID / 32] a
                                        bit per grid cell that holds a range query */
    uint32_t f_bits;
    double x0, y0, ix, iy;           /* the map's corner and cells per degree */
    stc_hit *hits;
    uint64_t cap;                    /* 0: counts only */
    unsigned long long *n_hits;
    unsigned long long *counts;
    uint32_t nq;
    uint32_t lds;                    /* nq <= QLDS: per-block counters in LDS */
    float fx[2], fy[2], fix, fiy;    /* range filter: the map's low corner in two parts, cells per degree */
};

#define QPIECE (8ull << 20) /* pinned bytes an upload goes through at a time */

/* host tables on their way to the device, as long as the batch makes them: built in pinned memory and sent with one copy
 * up to QPIECE, in pieces of that beyond (their sources stay as they are until then). Where no pinned memory is to be had
 * they go as they are. */
struct QueryUpload {
    uint8_t *host = nullptr, *dev = nullptr;
    uint64_t host_cap = 0, cap = 0, used = 0;
    bool pieces = false, lent = false; /* lent: host is part of QueryBufs::first */
    struct Table { const uint8_t *src; uint64_t at, bytes; }; /* src null: zeros */
    std::vector<Table> tables;
    /* device bytes that begin(bytes) would add */
    uint64_t growth(uint64_t bytes) const { return bytes <= cap ? 0 : room_for(bytes); }
    /* room for `bytes`, and nothing in it */
    int begin(uint64_t bytes) {
        used = 0;
        tables.clear();
        pieces = bytes > QPIECE;
        const uint64_t hc = std::min<uint64_t>(room_for(bytes), QPIECE);
        if (bytes > cap) {
            if (dev) (void)hipFree(dev);
            dev = nullptr;
            cap = 0;
            if (hipMalloc((void **)&dev, room_for(bytes)) != hipSuccess) {
                dev = nullptr;
                return -1;
            }
            cap = room_for(bytes);
        }
        if (std::min<uint64_t>(bytes, QPIECE) > host_cap) {
            free_host();
            if (hipHostMalloc((void **)&host, hc, hipHostMallocDefault) == hipSuccess) {
                host_cap = hc;
            } else {
                host = nullptr;
                pieces = true;
                (void)hipGetLastError();
            }
        }
        return 0;
    }
    static uint64_t room(uint64_t bytes) { return (bytes + 15) & ~15ull; }
    static uint64_t room_for(uint64_t bytes) { return bytes + bytes / 2 + 4096; }
    /* a table of n (from src, or zeros), and where it will be on the device */
    template <typename T>
    T *put(const T *src, uint64_t n) {
        T *d = (T *)(dev + used);
        if (pieces) tables.push_back(Table{(const uint8_t *)src, used, n * sizeof(T)});
        else if (src) memcpy(host + used, src, n * sizeof(T));
        else memset(host + used, 0, n * sizeof(T));
        used += room(n * sizeof(T));
        return d;
    }
    hipError_t send(hipStream_t s) {
        if (!pieces) return hipMemcpyAsync(dev, host, used, hipMemcpyHostToDevice, s);
        for (const Table &t : tables)
            for (uint64_t o = 0, n; o < t.bytes; o += n) {
                n = std::min<uint64_t>(host ? host_cap : t.bytes, t.bytes - o);
                if (host && t.src) memcpy(host, t.src + o, n);
                else if (host) memset(host, 0, n);
                hipError_t e = host || t.src ? hipMemcpyAsync(dev + t.at + o, host ? host : t.src + o, n, hipMemcpyHostToDevice, s)
                                             : hipMemsetAsync(dev + t.at, 0, n, s);
                if (e == hipSuccess) e = hipStreamSynchronize(s);
                if (e != hipSuccess) return e;
            }
        return hipSuccess;
    }
    void free_host() {
        if (host && !lent) (void)hipHostFree(host);
        host = nullptr;
        host_cap = 0;
        lent = false;
    }
    void release() {
        free_host();
        if (dev) (void)hipFree(dev);
        dev = nullptr;
        cap = 0;
    }
};

struct QueryBufs {
    QueryUpload batch, runs;         /* the batch's tables and zeroed counters; the runs and their candidates */
    uint64_t *res = nullptr;         /* pinned: the counters, then the first hits */
    uint64_t res_cap = 0;
    uint8_t *first = nullptr;        /* pinned: the two uploads' and res's first room in one (a block each is 250 us to free) */
    bool res_lent = false;
    void free_res() {
        if (res && !res_lent) (void)hipHostFree(res);
        res = nullptr;
        res_cap = 0;
        res_lent = false;
    }
    stc_hit *hits = nullptr;
    uint64_t hits_cap = 0;
    uint8_t *sort = nullptr;         /* keys and places of the hits, and the sort's scratch */
    uint64_t sort_cap = 0;
    stc_hit *out[2] = {nullptr, nullptr}; /* pinned: sorted hits on their way to the caller, a chunk each */
    hipEvent_t out_ev[2] = {nullptr, nullptr};
    uint32_t *wide = nullptr;        /* pinned: a hit's field did not fit its key bits */
};

#define QFETCH 65536u /* hits of a chunk */
#define QSORT_HOST 256u /* up to this many hits come with the counters and are sorted by the host: the device's ranking
                         * costs a wait more (some 30 us; the host takes about 80 at 1,000 hits) */
#define QRANK 16384u    /* and up to this many are ranked by comparing all with all */


void stc_query_bufs_free(QueryBufs *b) {
    if (!b) return;
    b->batch.release();
    b->runs.release();
    b->free_res();
    if (b->first) (void)hipHostFree(b->first);
    if (b->hits) (void)hipFree(b->hits);
    if (b->sort) (void)hipFree(b->sort);
    for (int i = 0; i < 2; i++) {
        if (b->out[i]) (void)hipHostFree(b->out[i]);
        if (b->out_ev[i]) (void)hipEventDestroy(b->out_ev[i]);
    }
    if (b->wide) (void)hipHostFree(b->wide);
    delete b;
}

template <typename T>
static int grow(T **p, uint64_t *cap, uint64_t need) {
    if (*p && *cap >= need) return 0;
    if (*p) (void)hipFree(*p);
    *p = nullptr;
    *cap = 0;
    uint64_t nc = std::max<uint64_t>(need + need / 2, 64);
    if (hipMalloc((void **)p, nc * sizeof(T)) != hipSuccess) {
        *p = nullptr;
        return -1;
    }
    *cap = nc;
    return 0;
}
/* with room for an ordinary batch, so that a context's first one allocates nothing */
QueryBufs *stc_query_bufs_new() {
    QueryBufs *b = new QueryBufs();
    const uint64_t batch = 100u << 10, runs = 50u << 10, res = (QSORT_HOST * 7 + 4096) * 8;
    if (hipHostMalloc((void **)&b->first, batch + runs + res, hipHostMallocDefault) == hipSuccess) {
        b->batch.host = b->first;
        b->batch.host_cap = batch;
        b->runs.host = b->first + batch;
        b->runs.host_cap = runs;
        b->res = (uint64_t *)(b->first + batch + runs);
        b->res_cap = res / 8;
        b->batch.lent = b->runs.lent = b->res_lent = true;
    } else {
        b->first = nullptr;
    }
    if (hipMalloc((void **)&b->batch.dev, batch) == hipSuccess) b->batch.cap = batch;
    if (hipMalloc((void **)&b->runs.dev, runs) == hipSuccess) b->runs.cap = runs;
    (void)grow(&b->hits, &b->hits_cap, 12u << 10);
    (void)hipGetLastError(); /* what could not be had now is asked for by the batch that needs it */
    return b;
}

/* The grid cell of a coordinate, the same arithmetic on the host (registration)
 * and the device (lookup). Any monotone map to cells serves: a meeting and a
 * query that intersect share the cell of the low corner of their intersection. */
__host__ __device__ inline int grid_cell(double v, double v0, double inv) {
    const double f = (v - v0) * inv;
    if (!(f >= 0.0)) return 0;
    if (f >= (double)QGRID) return QGRID - 1;
    return (int)f;
}

__host__ __device__ inline uint32_t oid_slot(uint32_t oid, uint32_t bits) {
    return (uint32_t)(((uint64_t)oid * 0x9E3779B97F4A7C15ull) >> (64 - bits));
}

/* the hit as the batch's next (all lanes that store together reserve at once: a
 * counter updated by every hit serialises on its address) */
__device__ inline void q_store(const QDev &Q, uint32_t qi, uint32_t pid, uint32_t target, uint32_t start, uint32_t end,
                               uint32_t source, const double *m) {
    if (!Q.cap || (Q.q[qi].flags & STC_QF_COUNT)) return;
    const uint64_t act = __ballot(1);
    const int lane = threadIdx.x & (STC_WAVE - 1), leader = __ffsll((long long)act) - 1;
    unsigned long long base = 0;
    if (lane == leader) base = atomicAdd(Q.n_hits, (unsigned long long)__popcll(act));
    base = __shfl(base, leader, STC_WAVE);
    const unsigned long long k = base + (unsigned long long)__popcll(act & ((1ull << lane) - 1ull));
    if (k < Q.cap) {
        stc_hit h;
        h.query = qi;
        h.pid = pid;
        h.target = target;
        h.start = start;
        h.end = end;
        h.source = source;
        h.mbr[0] = m[0];
        h.mbr[1] = m[1];
        h.mbr[2] = m[2];
        h.mbr[3] = m[3];
        Q.hits[k] = h;
    }
}

/* A scan's LDS: the per-block query counters (cleared on entry, added to the
 * global counts on exit: one atomic per query and block instead of one per
 * hit), then the batch's filter: 2^f_bits bits of id hashes and a bit per grid
 * cell, which turn away nearly every meeting no query asks for without a read
 * of the tables, and with range queries a bit per cell of a finer grid, of the
 * cells at and around their boxes. The launch sizes it (q_scan_lds). */
extern __shared__ uint32_t q_lds[];

__device__ inline uint32_t *q_scan_begin(const QDev &Q) {
    uint32_t *flt = q_lds + (Q.lds ? Q.nq : 0u);
    if (Q.lds)
        for (uint32_t i = threadIdx.x; i < Q.nq; i += blockDim.x) q_lds[i] = 0;
    const uint32_t words = (1u << Q.f_bits) / 32 + QGRID * QGRID / 32 + (Q.n_range ? QFINE * QFINE / 32 : 0);
    for (uint32_t i = threadIdx.x; i < words; i += blockDim.x) flt[i] = Q.filter[i];
    __syncthreads();
    return flt;
}
__device__ inline void q_scan_end(const QDev &Q) {
    __syncthreads();
    if (Q.lds)
        for (uint32_t i = threadIdx.x; i < Q.nq; i += blockDim.x)
            if (q_lds[i]) atomicAdd(&Q.counts[i], (unsigned long long)q_lds[i]);
}

/* A wave's hits on their way out, in LDS. A reservation per group of lanes that
 * hit together was an update of one address every few hits, 4 ns each in a
 * row, which bounded the scans of crowded boxes. */
struct QStage {
    stc_hit *h;
    uint32_t *n;
};

template <bool STORE = true>
__device__ inline void q_emit(const QDev &Q, const QStage &st, uint32_t qi, uint32_t pid, uint32_t target, uint32_t start,
                              uint32_t end, uint32_t source, const double *m) {
    if (Q.lds) atomicAdd(&q_lds[qi], 1u);
    else atomicAdd(&Q.counts[qi], 1ull);
    if (!STORE || !Q.cap || (Q.q[qi].flags & STC_QF_COUNT)) return;
    const uint32_t at = atomicAdd(st.n, 1u);
    if (at < QSTAGE) st.h[at] = stc_hit{qi, pid, target, start, end, source, {m[0], m[1], m[2], m[3]}};
    else q_store(Q, qi, pid, target, start, end, source, m);
}

/* n staged hits to the batch's hits from `base` on, by a wave */
__device__ inline void q_stage_out(const QDev &Q, const QStage &st, uint32_t n, unsigned long long base) {
    constexpr uint32_t W = sizeof(stc_hit) / 8;
    const uint64_t keep = base < Q.cap ? min<uint64_t>(n, Q.cap - base) : 0;
    uint64_t *dst = (uint64_t *)(Q.hits + base);
    const uint64_t *src = (const uint64_t *)st.h;
    for (uint32_t i = threadIdx.x & (STC_WAVE - 1); i < keep * W; i += STC_WAVE) dst[i] = src[i];
}

/* all lanes of the wave: its hits out where half its room is taken */
__device__ inline void q_stage_drain(const QDev &Q, const QStage &st) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const uint32_t n = (uint32_t)__builtin_amdgcn_readfirstlane((int)*(volatile uint32_t *)st.n);
    if (n < QSTAGE / 2) return;
    const uint32_t k = min(n, (uint32_t)QSTAGE);
    unsigned long long base = 0;
    if ((threadIdx.x & (STC_WAVE - 1)) == 0) base = atomicAdd(Q.n_hits, (unsigned long long)k);
    base = __shfl(base, 0, STC_WAVE);
    q_stage_out(Q, st, k, base);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    *(volatile uint32_t *)st.n = 0;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

/* the workgroup's last hits, one reservation; n: its waves' counts */
__device__ inline void q_stage_end(const QDev &Q, const QStage &st, const uint32_t *n) {
    __shared__ unsigned long long base;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t all = 0;
        for (uint32_t w = 0; w < blockDim.x / STC_WAVE; w++) all += min(n[w], (uint32_t)QSTAGE);
        base = all ? atomicAdd(Q.n_hits, (unsigned long long)all) : 0ull;
    }
    __syncthreads();
    unsigned long long b = base;
    const uint32_t wv = threadIdx.x / STC_WAVE;
    for (uint32_t w = 0; w < wv; w++) b += min(n[w], (uint32_t)QSTAGE);
    q_stage_out(Q, st, min(n[wv], (uint32_t)QSTAGE), b);
}

/* the workgroup's stages; without `on` (no hit is stored) only their shape */
#define Q_STAGE(st, on)                                                       \
    __shared__ stc_hit st##_h[(on) ? 256 / STC_WAVE : 1][(on) ? QSTAGE : 1];  \
    __shared__ uint32_t st##_n[256 / STC_WAVE];                               \
    const QStage st{st##_h[(on) ? threadIdx.x / STC_WAVE : 0], st##_n + threadIdx.x / STC_WAVE}; \
    if ((threadIdx.x & (STC_WAVE - 1)) == 0) *st.n = 0;                       \
    __syncthreads()

__device__ inline bool q_time(const stc_query &q, uint32_t s, uint32_t e) { return s <= q.t1 && e >= q.t0; }
__device__ inline bool q_box(const stc_query &q, const double *m) {
    return m[0] <= q.box[2] && m[2] >= q.box[0] && m[1] <= q.box[3] && m[3] >= q.box[1];
}

/* may an object or pair query name pid? */
__device__ inline bool q_may_oid(const QDev &Q, const uint32_t *flt, uint32_t pid) {
    const uint32_t h = oid_slot(pid, Q.f_bits);
    return (flt[h >> 5] >> (h & 31)) & 1u;
}

/* may a range query reach a box? In 32 bits: the low corner's cell of the fine
 * grid comes within a thousandth of a cell, and the filter's bits are those of
 * the cells that a query's box covers and of their neighbours, so a box of up
 * to half a cell is never missed; a larger one (or NaN) passes. */
__device__ inline int fine_cell(float v, const float *v0, float inv) {
    const float f = ((v - v0[0]) - v0[1]) * inv;
    if (!(f >= 0.0f)) return 0;
    return f >= (float)QFINE ? QFINE - 1 : (int)f;
}
__device__ inline bool q_may_box(const QDev &Q, const uint32_t *flt, float lo0, float lo1, float hi0, float hi1) {
    if (!((hi0 - lo0) * Q.fix <= 0.5f && (hi1 - lo1) * Q.fiy <= 0.5f)) return true;
    const uint32_t *fine = flt + (1u << Q.f_bits) / 32 + QGRID * QGRID / 32;
    const uint32_t cell = (uint32_t)(fine_cell(lo1, Q.fy, Q.fiy) * QFINE + fine_cell(lo0, Q.fx, Q.fix));
    return (fine[cell >> 5] >> (cell & 31)) & 1u;
}

/* the object and pair queries that name pid: the first of their list, -1 when there are none */
__device__ inline int32_t oid_queries(const QDev &Q, uint32_t pid) {
    const uint32_t mask = (1u << Q.oh_bits) - 1u;
    uint32_t h = oid_slot(pid, Q.oh_bits);
    for (;;) {
        uint32_t k = Q.oh_key[h];
        if (k == pid) return Q.oh_head[h];
        if (k == 0xFFFFFFFFu) return -1;
        h = (h + 1) & mask;
    }
}

/* the queries of that list for one meeting seen from pid */
template <bool STORE = true>
__device__ inline void match_oid(const QDev &Q, const QStage &st, int32_t qi, uint32_t pid, uint32_t target, uint32_t s,
                                 uint32_t e, uint32_t src, const double *m) {
    for (; qi >= 0; qi = Q.q_next[qi]) {
        const stc_query &q = Q.q[qi];
        if (!q_time(q, s, e)) continue;
        if (q.kind == STC_Q_OID || (q.kind == STC_Q_PAIR && q.oid2 == target))
            q_emit<STORE>(Q, st, (uint32_t)qi, pid, target, s, e, src, m);
    }
}

/* range queries of one meeting (called once per meeting) */
template <bool STORE = true>
__device__ inline void match_range(const QDev &Q, const QStage &st, const uint32_t *flt, uint32_t pid, uint32_t target, uint32_t s,
                                   uint32_t e, uint32_t src, const double *m) {
    const uint32_t *cells = flt + (1u << Q.f_bits) / 32;
    const int cx0 = grid_cell(m[0], Q.x0, Q.ix), cx1 = grid_cell(m[2], Q.x0, Q.ix);
    const int cy0 = grid_cell(m[1], Q.y0, Q.iy), cy1 = grid_cell(m[3], Q.y0, Q.iy);
    const bool one = cx0 == cx1 && cy0 == cy1;
    for (int cy = cy0; cy <= cy1; cy++)
        for (int cx = cx0; cx <= cx1; cx++) {
            const uint32_t cell = (uint32_t)(cy * QGRID + cx);
            if (!((cells[cell >> 5] >> (cell & 31)) & 1u)) continue;
            for (uint32_t j = Q.g_start[cell]; j < Q.g_start[cell + 1]; j++) {
                const uint32_t qi = Q.g_list[j];
                const stc_query &q = Q.q[qi];
                if (!q_time(q, s, e) || !q_box(q, m)) continue;
                if (!one && (grid_cell(fmax(m[0], q.box[0]), Q.x0, Q.ix) != cx || grid_cell(fmax(m[1], q.box[1]), Q.y0, Q.iy) != cy))
                    continue; /* counted in the cell of the intersection's low corner */
                q_emit<STORE>(Q, st, qi, pid, target, s, e, src, m);
            }
        }
}

/* CTF::ctf_get_key_oid, parse_key and new_parse_mbr (step_merge.cpp:325-379)
 * on the little-endian packed key at p. A key is read as two 8-byte words
 * wherever it starts (global memory takes unaligned reads; byte by byte a key
 * is 13 or 14 of them), so up to 15 bytes past its end: the packed keys of a
 * run are followed in their allocation by its CTF metadata. */
__device__ inline unsigned __int128 load_packed(const uint8_t *p, uint32_t kb) {
    uint64_t w[2];
    __builtin_memcpy(w, p, 16);
    if (kb < 8) {
        w[0] &= (1ull << (8 * kb)) - 1;
        w[1] = 0;
    } else if (kb < 16) {
        w[1] &= (1ull << (8 * (kb - 8))) - 1;
    }
    return ((unsigned __int128)w[1] << 64) | w[0];
}

__device__ inline uint32_t packed_pid(const stc_ctf_meta &c, unsigned __int128 k) {
    return (uint32_t)((k >> (c.id_bit + c.duration_bit + c.end_bit + c.mbr_bit)) & ((1ull << c.id_bit) - 1));
}

__device__ inline void decode_packed(const stc_ctf_meta &c, unsigned __int128 k, uint32_t *pid, uint32_t *target,
                                     uint32_t *start, uint32_t *end, double *box) {
    uint64_t vm = (uint64_t)(k & (((unsigned __int128)1 << c.mbr_bit) - 1));
    unsigned __int128 r = k >> c.mbr_bit;
    uint32_t e = (uint32_t)(r & ((1ull << c.end_bit) - 1));
    r >>= c.end_bit;
    uint32_t d = (uint32_t)(r & ((1ull << c.duration_bit) - 1));
    r >>= c.duration_bit;
    *target = (uint32_t)(r & ((1ull << c.id_bit) - 1));
    r >>= c.id_bit;
    *pid = (uint32_t)(r & ((1ull << c.id_bit) - 1));
    *end = e + c.end_time_min;
    *start = *end - d;
    const uint64_t mask_edge = (1ull << c.edge_bit) - 1, mask_low_y = (1ull << c.low_y_bit) - 1,
                   mask_low_x = (1ull << c.low_x_bit) - 1;
    uint64_t y = vm & mask_edge;
    vm >>= c.edge_bit;
    uint64_t x = vm & mask_edge;
    vm >>= c.edge_bit;
    uint64_t low1 = vm & mask_low_y;
    vm >>= c.low_y_bit;
    uint64_t low0 = vm & mask_low_x;
    const float w0 = c.mbr[2] - c.mbr[0], w1 = c.mbr[3] - c.mbr[1];
    const float longer = w0 > w1 ? w0 : w1;
    box[0] = (double)c.mbr[0] + (double)low0 / (double)mask_low_x * (double)w0;
    box[1] = (double)c.mbr[1] + (double)low1 / (double)mask_low_y * (double)w1;
    box[2] = box[0] + (double)x / (double)mask_edge * (double)longer;
    box[3] = box[1] + (double)y / (double)mask_edge * (double)longer;
}

__device__ inline void decode_tail(const uint64_t *o_keys, const float4 *o_boxes, uint32_t i, uint32_t base,
                                   uint32_t *pid, uint32_t *target, uint32_t *start, uint32_t *end, double *m) {
    uint64_t lo = o_keys[2 * i], hi = o_keys[2 * i + 1];
    *pid = (uint32_t)(hi >> 26) & MASK26;
    *target = (uint32_t)hi & MASK26;
    *end = (uint32_t)lo + base;
    *start = *end - (uint32_t)(lo >> 32);
    float4 b = o_boxes[i];
    m[0] = b.x;
    m[1] = b.y;
    m[2] = b.z;
    m[3] = b.w;
}

/* One read of the live meetings, several at once so that no read waits for
 * another: the ids for object queries, the boxes for range queries. A meeting
 * that the filters let pass waits in the wave's LDS until 64 of them are looked
 * up together: nearly every wave has one or two in every round, and the
 * lookup's chain of reads for those few was what bounded the scan. With 28-byte
 * meetings read whole or looked up one by one: 1,000 objects among 256M
 * meetings 2.10 -> 0.83 ms (8 bytes each at 2.5 TB/s; the id filter and the
 * table now bound it), one among 10M 52 -> 25 us, 48 crowded boxes with 446,000
 * hits 465 -> 257 us (with the hits' reservations, at q_emit).
 * Where ranges are counted, or asked among ids, most of the time goes to the
 * lookups, whose reads the waves in flight have to hide. The round's meetings
 * all go to the list before any is looked up (AFTER), so that the lookup is in
 * the code once and runs with their boxes out of the registers, and a batch
 * that stores no hit (STORE) has no stage for them: 82 to 86 registers, five
 * waves a SIMD and 15 KB of LDS a workgroup become 61 and 16, or 48 (eight
 * waves) and 3. 8.6M meetings: 100 counted boxes of 50 to 500 m where people
 * are 362 -> 316 us, 20,000 of them 26.1 -> 23.1 ms, 256 of the whole map
 * 19.9 -> 17.6 (28-byte meetings looked up as they came: 351 us, 23.9 and
 * 17.4 ms), 128 mixed queries 576 -> 540 us. Counting batches read two
 * meetings a lane at a time (one small box: 166 us; four 171, eight 190).
 * The lookup stays inside the round with ids alone, where few meetings pass and
 * it is short (1,000 ids: 167 us, 176 after it), and for stored ranges alone,
 * bound by their hits (1,000 boxes, a thousand hits kept: 5.30 ms, 5.41). */
template <bool OIDS, bool RANGES, bool STORE>
__global__ __launch_bounds__(256) void k_q_live(Meets t, uint64_t nb, uint32_t last_t, QDev Q) {
    constexpr int U = RANGES ? (STORE ? 4 : 2) : 8;
    constexpr bool AFTER = RANGES && (OIDS || !STORE); /* lookups after the round */
    __shared__ uint32_t wait[256 / STC_WAVE][(AFTER ? U + 1 : 2) * STC_WAVE];
    const uint32_t *flt = q_scan_begin(Q);
    Q_STAGE(st, STORE);
    uint32_t *wq = wait[threadIdx.x / STC_WAVE];
    uint32_t waiting = 0;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    const uint64_t first = (uint64_t)blockIdx.x * blockDim.x + (threadIdx.x & ~(STC_WAVE - 1u));
    const uint32_t lane = threadIdx.x & (STC_WAVE - 1);
    const uint64_t lt = (1ull << lane) - 1ull;
    auto look_up = [&](uint32_t n) { /* the last n of the waiting */
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        waiting -= n;
        if (lane < n) {
            const uint64_t i = wq[waiting + lane]; /* a step has fewer than 2^32 meetings */
            const Bucket b = t.at(i);
            const uint32_t a = (uint32_t)(b.key >> 32), c = (uint32_t)b.key;
            if (c != DEAD_B) {
                const double m[4] = {o2f(b.mbr[0]), o2f(b.mbr[1]), o2f(b.mbr[2]), o2f(b.mbr[3])};
                /* a live meeting ends at the step that built the arrays */
                if constexpr (OIDS) {
                    match_oid<STORE>(Q, st, oid_queries(Q, a), a, c, b.start, last_t, 0, m);
                    match_oid<STORE>(Q, st, oid_queries(Q, c), c, a, b.start, last_t, 0, m);
                }
                if constexpr (RANGES) match_range<STORE>(Q, st, flt, a, c, b.start, last_t, 0, m);
            }
        }
        if constexpr (STORE) q_stage_drain(Q, st);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); /* the list's places are written again */
        __builtin_amdgcn_wave_barrier();
    };
    for (uint64_t i0 = first;; i0 += stride * U) {
        const bool end = i0 >= nb;
        if (!end) {
            unsigned long long key[U];
            uint4 mbr[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint64_t i = min(i0 + lane + u * stride, nb - 1);
                if constexpr (OIDS) key[u] = t.key(i);
                if constexpr (RANGES) mbr[u] = t.mbr(i);
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint64_t i = i0 + lane + u * stride;
                bool pass = false;
                if constexpr (RANGES) pass = q_may_box(Q, flt, o2f(mbr[u].x), o2f(mbr[u].y), o2f(mbr[u].z), o2f(mbr[u].w));
                if constexpr (OIDS) {
                    pass = pass || q_may_oid(Q, flt, (uint32_t)(key[u] >> 32)) || q_may_oid(Q, flt, (uint32_t)key[u]);
                    pass = pass && (uint32_t)key[u] != DEAD_B;
                }
                pass = pass && i < nb;
                const uint64_t passing = __ballot(pass);
                if (pass) wq[waiting + (uint32_t)__popcll(passing & lt)] = (uint32_t)i;
                waiting += (uint32_t)__popcll(passing);
                if constexpr (!AFTER)
                    if (waiting >= STC_WAVE) look_up(STC_WAVE);
            }
        }
        while (waiting >= (end ? 1u : (uint32_t)STC_WAVE)) look_up(min(waiting, (uint32_t)STC_WAVE));
        if (end) break;
    }
    if constexpr (STORE) q_stage_end(Q, st, st_n);
    q_scan_end(Q);
}

__global__ __launch_bounds__(256) void k_q_mem(const uint64_t *__restrict__ keys, const float4 *__restrict__ boxes,
                                               uint64_t n, uint32_t base, QDev Q) {
    const uint32_t *flt = q_scan_begin(Q);
    Q_STAGE(st, true);
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    const uint64_t first = (uint64_t)blockIdx.x * blockDim.x + (threadIdx.x & ~(STC_WAVE - 1u)), lane = threadIdx.x & (STC_WAVE - 1);
    for (uint64_t i0 = first; i0 < n; i0 += stride) {
        const uint64_t i = i0 + lane;
        if (i < n) {
            const uint64_t hi = keys[2 * i + 1];
            const uint32_t pid = (uint32_t)(hi >> 26) & MASK26, target = (uint32_t)hi & MASK26;
            float4 b = make_float4(0, 0, 0, 0);
            if (Q.n_range) b = boxes[i];
            const int32_t qo = Q.oh_bits && q_may_oid(Q, flt, pid) ? oid_queries(Q, pid) : -1;
            const bool mr = Q.n_range && pid < target && q_may_box(Q, flt, b.x, b.y, b.z, b.w);
            if (qo >= 0 || mr) {
                uint32_t p, c, start, end;
                double m[4];
                decode_tail(keys, boxes, (uint32_t)i, base, &p, &c, &start, &end, m);
                match_oid(Q, st, qo, pid, target, start, end, 1, m);
                if (mr) match_range(Q, st, flt, pid, target, start, end, 1, m);
            }
        }
        q_stage_drain(Q, st);
    }
    q_stage_end(Q, st, st_n);
    q_scan_end(Q);
}

/* one query's hits counted by the lanes, added to its count at once */
__device__ inline void q_count_wave(const QDev &Q, uint32_t qi, uint32_t mine) {
    for (int o = STC_WAVE / 2; o > 0; o >>= 1) mine += __shfl_down(mine, o, STC_WAVE);
    if ((threadIdx.x & (STC_WAVE - 1)) == 0 && mine) atomicAdd(&Q.counts[qi], (unsigned long long)mine);
}

/* Object and pair queries against the runs, a wave per (query, run): the
 * object's CTF by its sid, the first of its packed keys by 64 probes a round
 * (two or three dependent reads; a thread's binary search took fifteen, of
 * fourteen bytes each: 18 us for one query, 5 now; 64 queries, 3 runs: 89 and 8), then its records 64
 * at a time; oversize objects (sid 1) scan the oversize buffer. */
__global__ __launch_bounds__(256) void k_q_run_oid(const QueryRunDev *__restrict__ runs, uint32_t nruns,
                                                   const uint32_t *__restrict__ oq, uint32_t noq, uint32_t n_objects,
                                                   QDev Q) {
    const int lane = threadIdx.x & (STC_WAVE - 1);
    const uint64_t g = (uint64_t)__builtin_amdgcn_readfirstlane((int)(((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / STC_WAVE));
    if (g >= (uint64_t)noq * nruns) return;
    const QueryRunDev R = runs[g / noq];
    const uint32_t qi = oq[g % noq];
    const stc_query q = Q.q[qi];
    if (q.oid >= n_objects) return;
    const uint16_t sid = R.sids[q.oid];
    uint32_t pid, target, start, end, found = 0;
    double m[4];
    if (sid == 0) return;
    if (sid == 1) {
        for (uint32_t i = (uint32_t)lane; i < R.n_tail; i += STC_WAVE) {
            decode_tail(R.o_keys, R.o_boxes, i, R.end_time_min, &pid, &target, &start, &end, m);
            if (pid != q.oid || !q_time(q, start, end)) continue;
            if (q.kind == STC_Q_OID || target == q.oid2) {
                found++;
                q_store(Q, qi, pid, target, start, end, R.source, m);
            }
        }
        q_count_wave(Q, qi, found);
        return;
    }
    const uint32_t c = sid - 2u;
    if (c >= R.ctf_count) return;
    const stc_ctf_meta ctf = R.ctfs[c];
    const uint32_t kb = ctf.key_bit / 8;
    const uint8_t *base = R.key_bytes + R.byte_base[c];
    uint32_t lo = 0, hi = ctf.kv_capacity; /* the first key not below the object's is in [lo, hi] */
    while (hi - lo > STC_WAVE) {
        const uint32_t step = (hi - lo) / STC_WAVE, at = lo + (uint32_t)lane * step + step - 1;
        const uint64_t below = __ballot(packed_pid(ctf, load_packed(base + (uint64_t)at * kb, kb)) < q.oid);
        const uint32_t k = below == ~0ull ? STC_WAVE : (uint32_t)__ffsll((long long)~below) - 1u;
        if (k < STC_WAVE) hi = lo + (k + 1) * step - 1;
        lo += k * step;
    }
    {
        const uint32_t at = lo + (uint32_t)lane;
        const bool below = at < hi && packed_pid(ctf, load_packed(base + (uint64_t)at * kb, kb)) < q.oid;
        lo += (uint32_t)__popcll(__ballot(below));
    }
    for (uint32_t i0 = lo; i0 < ctf.kv_capacity; i0 += STC_WAVE) {
        const uint32_t i = i0 + (uint32_t)lane;
        unsigned __int128 k = 0;
        bool own = false;
        if (i < ctf.kv_capacity) {
            k = load_packed(base + (uint64_t)i * kb, kb);
            own = packed_pid(ctf, k) == q.oid;
        }
        const uint64_t run = __ballot(own);
        /* the object's records end at the first key that is not its own */
        const uint32_t len = run == ~0ull ? STC_WAVE : (uint32_t)__ffsll((long long)~run) - 1u;
        if ((uint32_t)lane < len) {
            decode_packed(ctf, k, &pid, &target, &start, &end, m);
            if (q_time(q, start, end) && (q.kind == STC_Q_OID || target == q.oid2)) {
                found++;
                q_store(Q, qi, pid, target, start, end, R.source, m);
            }
        }
        if (len < STC_WAVE) break;
    }
    q_count_wave(Q, qi, found);
}

/* range queries: one block per (query, run, CTF) candidate; CTF 0xFFFFFFFF is
 * the run's oversize buffer */
__global__ __launch_bounds__(256) void k_q_run_range(const QueryRunDev *__restrict__ runs,
                                                     const uint4 *__restrict__ cand, QDev Q) {
    const uint4 cd = cand[blockIdx.x];
    const uint32_t qi = cd.x;
    const stc_query q = Q.q[qi];
    const QueryRunDev R = runs[cd.y];
    uint32_t pid, target, start, end, found = 0;
    double m[4];
    Q_STAGE(st, true);
    const bool store = Q.cap && !(q.flags & STC_QF_COUNT);
    auto hit = [&]() {
        found++;
        if (!store) return;
        const uint32_t at = atomicAdd(st.n, 1u);
        if (at < QSTAGE) st.h[at] = stc_hit{qi, pid, target, start, end, R.source, {m[0], m[1], m[2], m[3]}};
        else q_store(Q, qi, pid, target, start, end, R.source, m);
    };
    const uint32_t first = threadIdx.x & ~(STC_WAVE - 1u), lane = threadIdx.x & (STC_WAVE - 1);
    if (cd.z == 0xFFFFFFFFu) {
        for (uint32_t i0 = first; i0 < R.n_tail; i0 += blockDim.x) {
            if (i0 + lane < R.n_tail) {
                decode_tail(R.o_keys, R.o_boxes, i0 + lane, R.end_time_min, &pid, &target, &start, &end, m);
                if (pid < target && q_time(q, start, end) && q_box(q, m)) hit();
            }
            if (store) q_stage_drain(Q, st);
        }
    } else {
        const stc_ctf_meta ctf = R.ctfs[cd.z];
        const uint32_t kb = ctf.key_bit / 8;
        const uint8_t *base = R.key_bytes + R.byte_base[cd.z];
        for (uint32_t i0 = first; i0 < ctf.kv_capacity; i0 += blockDim.x) {
            if (i0 + lane < ctf.kv_capacity) {
                decode_packed(ctf, load_packed(base + (uint64_t)(i0 + lane) * kb, kb), &pid, &target, &start, &end, m);
                if (pid < target && q_time(q, start, end) && q_box(q, m)) hit();
            }
            if (store) q_stage_drain(Q, st);
        }
    }
    if (store) q_stage_end(Q, st, st_n);
    q_count_wave(Q, qi, found);
}

/* one block per CTF: exact union box, time span and forward-record count */
#define STATS_CHUNK 4096u /* records of a CTF one block summarises */

/* one block per (CTF, chunk of STATS_CHUNK records): a partial summary,
 * combined per CTF on the host */
__global__ __launch_bounds__(256) void k_ctf_stats(QueryRunDev R, const uint2 *__restrict__ items,
                                                   CtfStats *out) {
    __shared__ double sb[4][256];
    __shared__ uint32_t su[4][256];
    const uint32_t c = items[blockIdx.x].x, first = items[blockIdx.x].y, tid = threadIdx.x;
    const stc_ctf_meta ctf = R.ctfs[c];
    const uint32_t kb = ctf.key_bit / 8;
    const uint8_t *base = R.key_bytes + R.byte_base[c];
    const uint32_t last = min(ctf.kv_capacity, first + STATS_CHUNK);
    double b0 = INFINITY, b1 = INFINITY, b2 = -INFINITY, b3 = -INFINITY;
    uint32_t smin = 0xFFFFFFFFu, emax = 0, fwd = 0, irregular = 0;
    for (uint32_t i = first + tid; i < last; i += blockDim.x) {
        uint32_t pid, target, start, end;
        double m[4];
        decode_packed(ctf, load_packed(base + (uint64_t)i * kb, kb), &pid, &target, &start, &end, m);
        if (!(m[0] <= m[2]) || !(m[1] <= m[3]) || start > end) irregular = 1; /* also catches NaN */
        b0 = fmin(b0, m[0]);
        b1 = fmin(b1, m[1]);
        b2 = fmax(b2, m[2]);
        b3 = fmax(b3, m[3]);
        smin = min(smin, start);
        emax = max(emax, end);
        fwd += pid < target;
    }
    sb[0][tid] = b0;
    sb[1][tid] = b1;
    sb[2][tid] = b2;
    sb[3][tid] = b3;
    su[0][tid] = smin;
    su[1][tid] = emax;
    su[2][tid] = fwd;
    su[3][tid] = irregular;
    __syncthreads();
    for (uint32_t o = blockDim.x / 2; o > 0; o >>= 1) {
        if (tid < o) {
            sb[0][tid] = fmin(sb[0][tid], sb[0][tid + o]);
            sb[1][tid] = fmin(sb[1][tid], sb[1][tid + o]);
            sb[2][tid] = fmax(sb[2][tid], sb[2][tid + o]);
            sb[3][tid] = fmax(sb[3][tid], sb[3][tid + o]);
            su[0][tid] = min(su[0][tid], su[0][tid + o]);
            su[1][tid] = max(su[1][tid], su[1][tid + o]);
            su[2][tid] += su[2][tid + o];
            su[3][tid] |= su[3][tid + o];
        }
        __syncthreads();
    }
    if (tid == 0) {
        CtfStats st;
        st.box[0] = sb[0][0];
        st.box[1] = sb[1][0];
        st.box[2] = sb[2][0];
        st.box[3] = sb[3][0];
        st.start_min = su[0][0];
        st.end_max = su[1][0];
        st.n_fwd = su[2][0];
        st.regular = !su[3][0];
        out[blockIdx.x] = st;
    }
}

static uint32_t blocks(uint64_t n, uint32_t b) { return (uint32_t)std::max<uint64_t>((n + b - 1) / b, 1); }

#define QCK(expr)                                                                                   \
    do {                                                                                            \
        hipError_t e_ = (expr);                                                                     \
        if (e_ != hipSuccess) return stc_hip_fail(e_, #expr, __FILE__, __LINE__);                   \
    } while (0)

/* CTF::new_parse_mbr_f_box: the double expressions of new_parse_mbr stored to
 * float, the high corner computed from the stored (float) low corner */
__device__ inline float4 decode_fbox(const stc_ctf_meta &c, uint64_t vm) {
    const uint64_t mask_edge = (1ull << c.edge_bit) - 1, mask_low_y = (1ull << c.low_y_bit) - 1,
                   mask_low_x = (1ull << c.low_x_bit) - 1;
    uint64_t y = vm & mask_edge;
    vm >>= c.edge_bit;
    uint64_t x = vm & mask_edge;
    vm >>= c.edge_bit;
    uint64_t low1 = vm & mask_low_y;
    vm >>= c.low_y_bit;
    uint64_t low0 = vm & mask_low_x;
    const float w0 = c.mbr[2] - c.mbr[0], w1 = c.mbr[3] - c.mbr[1];
    const float longer = w0 > w1 ? w0 : w1;
    float4 b;
    b.x = (float)((double)c.mbr[0] + (double)low0 / (double)mask_low_x * (double)w0);
    b.y = (float)((double)c.mbr[1] + (double)low1 / (double)mask_low_y * (double)w1);
    b.z = (float)((double)b.x + (double)x / (double)mask_edge * (double)longer);
    b.w = (float)((double)b.y + (double)y / (double)mask_edge * (double)longer);
    return b;
}

/* A run's records are grouped by object, so the lanes of a wave mostly share
 * a few objects: the first lane of each run of equal ids adds up the run's
 * length (64 updates of one address would be serialised), and its lanes take
 * the records' places among their objects' from there. */
__global__ __launch_bounds__(256) void k_compact_decode(QueryRunDev R, uint64_t kv_count, uint32_t num_objects,
                                                        uint32_t base, uint64_t out0, uint64_t *__restrict__ keys,
                                                        float4 *__restrict__ boxes, uint32_t *__restrict__ same_pid_count,
                                                        uint32_t *__restrict__ ord, uint32_t *__restrict__ bad) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & (STC_WAVE - 1);
    uint32_t pid = 0xFFFFFFFFu; /* no object: lanes past the end and bad records */
    if (i < kv_count + R.n_tail) {
        uint32_t p, target, dur, end;
        float4 b;
        if (i < kv_count) {
            /* the record's CTF: the last c with rec_base[c] <= i */
            uint32_t lo = 0, hi = R.ctf_count;
            while (hi - lo > 1) {
                uint32_t mid = (lo + hi) / 2;
                if (R.rec_base[mid] <= i) lo = mid;
                else hi = mid;
            }
            const stc_ctf_meta c = R.ctfs[lo];
            const uint32_t kb = c.key_bit / 8;
            unsigned __int128 k = load_packed(R.key_bytes + R.byte_base[lo] + (i - R.rec_base[lo]) * kb, kb);
            const uint64_t vm = (uint64_t)(k & (((unsigned __int128)1 << c.mbr_bit) - 1));
            unsigned __int128 r = k >> c.mbr_bit;
            end = (uint32_t)(r & ((1ull << c.end_bit) - 1)) + c.end_time_min;
            r >>= c.end_bit;
            dur = (uint32_t)(r & ((1ull << c.duration_bit) - 1));
            r >>= c.duration_bit;
            target = (uint32_t)(r & ((1ull << c.id_bit) - 1));
            r >>= c.id_bit;
            p = (uint32_t)(r & ((1ull << c.id_bit) - 1));
            b = decode_fbox(c, vm);
        } else {
            const uint64_t j = i - kv_count;
            const uint64_t lo = R.o_keys[2 * j], hi = R.o_keys[2 * j + 1];
            p = (uint32_t)(hi >> 26) & MASK26;
            target = (uint32_t)hi & MASK26;
            end = (uint32_t)lo + R.end_time_min;
            dur = (uint32_t)(lo >> 32);
            b = R.o_boxes[j];
        }
        keys[2 * (out0 + i)] = ((uint64_t)dur << 32) | (uint32_t)(end - base);
        keys[2 * (out0 + i) + 1] = ((uint64_t)p << 26) | target;
        boxes[out0 + i] = b;
        if (p >= num_objects || target >= num_objects) { /* not a key this context wrote */
            atomicOr(bad, 1u);
        } else {
            pid = p;
        }
    }
    const uint32_t prev = __shfl_up(pid, 1, STC_WAVE);
    const bool head = lane == 0 || prev != pid;
    const uint64_t heads = __ballot(head), upto = heads & (~0ull >> (STC_WAVE - 1 - lane));
    const int first = STC_WAVE - 1 - __clzll((long long)upto);
    const uint64_t after = lane == STC_WAVE - 1 ? 0ull : heads >> (lane + 1);
    uint32_t at = 0;
    if (head && pid != 0xFFFFFFFFu)
        at = atomicAdd(&same_pid_count[pid], after ? (uint32_t)__ffsll((long long)after) : (uint32_t)(STC_WAVE - lane));
    at = (uint32_t)__shfl((int)at, first, STC_WAVE) + (uint32_t)(lane - first);
    if (pid != 0xFFFFFFFFu) ord[out0 + i] = at;
}

__global__ void k_compact_sids(const uint16_t *__restrict__ run_sids, uint32_t n, uint16_t *__restrict__ sids) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && run_sids[i] == 1) sids[i] = 1;
}

int stc_compact_decode(const QueryRunDev &R, uint64_t kv_count, uint32_t num_objects, uint32_t base, uint64_t out0,
                       uint64_t *keys, float4 *boxes, uint32_t *same_pid_count, uint32_t *ord, uint16_t *sids,
                       uint32_t *bad, hipStream_t s) {
    if (kv_count + R.n_tail)
        hipLaunchKernelGGL(k_compact_decode, dim3(blocks(kv_count + R.n_tail, 256)), dim3(256), 0, s, R, kv_count,
                           num_objects, base, out0, keys, boxes, same_pid_count, ord, bad);
    QCK(hipGetLastError());
    hipLaunchKernelGGL(k_compact_sids, dim3(blocks(num_objects, 256)), dim3(256), 0, s, R.sids, num_objects, sids);
    QCK(hipGetLastError());
    return STC_OK;
}

int stc_query_ctf_stats(const QueryRunDev &run, const stc_ctf_meta *host_ctfs, std::vector<CtfStats> &out,
                        hipStream_t s) {
    out.assign(run.ctf_count, CtfStats());
    if (!run.ctf_count) return STC_OK;
    /* work items: every CTF in chunks of STATS_CHUNK records (an empty CTF still gets one) */
    std::vector<uint2> items;
    std::vector<uint32_t> first_item(run.ctf_count);
    for (uint32_t c = 0; c < run.ctf_count; c++) {
        first_item[c] = (uint32_t)items.size();
        const uint32_t cap = host_ctfs[c].kv_capacity;
        for (uint32_t k = 0; k == 0 || k < cap; k += STATS_CHUNK) items.push_back(make_uint2(c, k));
    }
    const uint32_t ni = (uint32_t)items.size();
    CtfStats *d = nullptr;
    uint2 *di = nullptr;
    QCK(hipMalloc((void **)&d, ni * sizeof(CtfStats)));
    hipError_t e = hipMalloc((void **)&di, ni * sizeof(uint2));
    std::vector<CtfStats> part(ni);
    if (e == hipSuccess) e = hipMemcpyAsync(di, items.data(), ni * sizeof(uint2), hipMemcpyHostToDevice, s);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_ctf_stats, dim3(ni), dim3(256), 0, s, run, (const uint2 *)di, d);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(part.data(), d, ni * sizeof(CtfStats), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    (void)hipFree(d);
    if (di) (void)hipFree(di);
    if (e != hipSuccess) return stc_hip_fail(e, "CTF statistics", __FILE__, __LINE__);
    for (uint32_t c = 0; c < run.ctf_count; c++) {
        const uint32_t k1 = c + 1 < run.ctf_count ? first_item[c + 1] : ni;
        CtfStats st = part[first_item[c]];
        for (uint32_t k = first_item[c] + 1; k < k1; k++) {
            const CtfStats &p = part[k];
            st.box[0] = std::fmin(st.box[0], p.box[0]);
            st.box[1] = std::fmin(st.box[1], p.box[1]);
            st.box[2] = std::fmax(st.box[2], p.box[2]);
            st.box[3] = std::fmax(st.box[3], p.box[3]);
            st.start_min = std::min(st.start_min, p.start_min);
            st.end_max = std::max(st.end_max, p.end_max);
            st.n_fwd += p.n_fwd;
            st.regular = st.regular && p.regular;
        }
        out[c] = st;
    }
    return STC_OK;
}

/* the counters and the first hits (at most `most`) to host memory: one launch, and the only wait of a small batch */
__global__ void k_q_finish(const unsigned long long *__restrict__ counters, uint32_t nq, const uint64_t *__restrict__ hits,
                           uint64_t most, uint64_t *__restrict__ out) {
    const uint64_t c = min<uint64_t>(counters[0], most), words = nq + 1ull + c * 7;
    for (uint64_t w = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; w < words; w += (uint64_t)gridDim.x * blockDim.x)
        out[w] = w <= nq ? counters[w] : hits[w - nq - 1];
}

/* ---------------- the hits in order ---------------- */

/* how a hit's (query, source, pid, target, start, end) is packed into sort keys */
struct HitKeyBits {
    uint32_t q, src, id, t; /* bits of a field */
    uint32_t two;           /* two keys: (query, source, pid) and (target, start, end); else one of all six */
};

/* the hits' sort keys, taken in the order idx when there is one; part 0: the low key or the only one, 1: the high key */
__global__ void k_hit_keys(const stc_hit *__restrict__ hits, const uint32_t *__restrict__ idx, uint32_t n, HitKeyBits b,
                           int part, uint64_t *__restrict__ keys, uint32_t *__restrict__ wide) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const stc_hit &h = hits[idx ? idx[i] : i];
    const uint64_t q = h.query, src = h.source, pid = h.pid, tgt = h.target, st = h.start, en = h.end;
    if ((q >> b.q) | (src >> b.src) | (pid >> b.id) | (tgt >> b.id) | (st >> b.t) | (en >> b.t)) *wide = 1;
    const uint64_t high = (((q << b.src) | src) << b.id) | pid, low = (((tgt << b.t) | st) << b.t) | en;
    keys[i] = part ? high : b.two ? low : (high << (b.id + 2 * b.t)) | low;
}

/* hits[idx[first ..]] to out (host memory), 8 bytes a thread */
__global__ void k_hit_gather(const uint64_t *__restrict__ hits, const uint32_t *__restrict__ idx, uint32_t first,
                             uint32_t words, uint64_t *__restrict__ out) {
    const uint32_t w = blockIdx.x * blockDim.x + threadIdx.x;
    if (w < words) out[w] = hits[(uint64_t)idx[first + w / 7] * 7 + w % 7];
}
static_assert(sizeof(stc_hit) == 56, "a hit is seven words");

/* rank[i] += the hits of the workgroup's tile that come before hit i: (query,
 * source, pid, target, start, end) as three words, equal ones in the order they
 * were found. A radix sort of a few thousand hits is some twenty launches and
 * nothing but latency; all with all is n^2 / 2^16 workgroups of 256 short
 * rounds (128 queries with some 3,000 hits: 714 -> 672 us, a step with 1,200
 * contacts 1,679 -> 1,646). */
__global__ __launch_bounds__(256) void k_hit_rank(const stc_hit *__restrict__ hits, uint32_t n, uint32_t *__restrict__ rank) {
    __shared__ uint64_t ka[256], kb[256], kc[256];
    const uint32_t i = blockIdx.x * 256 + threadIdx.x, j0 = blockIdx.y * 256, j = j0 + threadIdx.x;
    auto load = [&](uint32_t k, uint64_t *a, uint64_t *b, uint64_t *c) {
        const stc_hit &h = hits[min(k, n - 1)];
        *a = (uint64_t)h.query << 32 | h.source;
        *b = (uint64_t)h.pid << 32 | h.target;
        *c = (uint64_t)h.start << 32 | h.end;
    };
    uint64_t a, b, c;
    load(j, &ka[threadIdx.x], &kb[threadIdx.x], &kc[threadIdx.x]);
    load(i, &a, &b, &c);
    __syncthreads();
    const uint32_t m = min(256u, n - j0);
    uint32_t before = 0;
#pragma unroll 4
    for (uint32_t k = 0; k < m; k++) {
        const uint64_t x = ka[k], y = kb[k], z = kc[k];
        const bool last = z < c || (z == c && j0 + k < i);
        before += (x < a || (x == a && (y < b || (y == b && last)))) ? 1u : 0u;
    }
    if (i < n && before) atomicAdd(&rank[i], before);
}

/* the hits to their ranks in out (host memory), 8 bytes a thread */
__global__ void k_hit_place(const uint64_t *__restrict__ hits, const uint32_t *__restrict__ rank, uint32_t words,
                            uint64_t *__restrict__ out) {
    const uint32_t w = blockIdx.x * blockDim.x + threadIdx.x;
    if (w < words) out[(uint64_t)rank[w / 7] * 7 + w % 7] = hits[w];
}

/* The n stored hits to the caller's `hits`, sorted by (query, source, pid,
 * target, start, end): up to QRANK of them ranked, more by a radix sort of the packed fields on the device, then
 * chunks gathered in order into pinned memory and copied out while the next is
 * gathered. *done stays false when the fields do not pack, a value does not fit
 * its bits, the scratch would leave less than `reserve` bytes of device memory,
 * or no pinned memory is to be had: the caller then sorts on the host. (330,000 hits: one host thread
 * sorted them in 17 ms; the sort takes 0.25 ms, the fetch is bound by the link and
 * the copy into the caller's memory.) */
static int fetch_sorted(QueryBufs *B, const QueryState &st, uint32_t nq, uint64_t n64, stc_hit *hits, uint64_t reserve,
                        bool *done, hipStream_t s) {
    *done = false;
    auto bits_for = [](uint64_t v) { uint32_t b = 1; while (b < 63 && (v >> b)) b++; return b; };
    HitKeyBits kb{bits_for(nq - 1), 1, bits_for(st.num_objects - 1), bits_for(st.last_t), 0};
    for (const QueryRunDev &r : st.runs) kb.src = std::max(kb.src, bits_for(r.source));
    const uint32_t hb = kb.q + kb.src + kb.id, lb = kb.id + 2 * kb.t;
    kb.two = hb + lb > 64;
    const bool ranked = n64 <= QRANK;
    if (!ranked && (n64 >= (1ull << 31) || hb > 64 || lb > 64)) return STC_OK;
    const uint32_t n = (uint32_t)n64;
    const uint64_t bytes = ranked ? n64 * 4 : n64 * 24 + stc_radix_temp_words(n) * 4;
    if (B->sort_cap < bytes) {
        size_t free_b = 0, total_b = 0;
        if (hipMemGetInfo(&free_b, &total_b) != hipSuccess || bytes + bytes / 2 + reserve > free_b + B->sort_cap) return STC_OK;
        if (grow(&B->sort, &B->sort_cap, bytes)) {
            (void)hipGetLastError(); /* the host sorts */
            return STC_OK;
        }
    }
    bool pinned = B->wide || hipHostMalloc((void **)&B->wide, sizeof(uint32_t), hipHostMallocDefault) == hipSuccess;
    for (int i = 0; i < 2 && pinned; i++) {
        pinned = B->out[i] || hipHostMalloc((void **)&B->out[i], QFETCH * sizeof(stc_hit), hipHostMallocDefault) == hipSuccess;
        if (!B->out_ev[i]) QCK(hipEventCreateWithFlags(&B->out_ev[i], hipEventDisableTiming));
    }
    if (!pinned) {
        (void)hipGetLastError(); /* the host sorts */
        return STC_OK;
    }
    if (ranked) {
        uint32_t *rank = (uint32_t *)B->sort;
        QCK(hipMemsetAsync(rank, 0, n * 4ull, s));
        hipLaunchKernelGGL(k_hit_rank, dim3(blocks(n, 256), blocks(n, 256)), dim3(256), 0, s, B->hits, n, rank);
        hipLaunchKernelGGL(k_hit_place, dim3(blocks(n * 7ull, 256)), dim3(256), 0, s, (const uint64_t *)B->hits,
                           (const uint32_t *)rank, n * 7, (uint64_t *)B->out[0]);
        QCK(hipGetLastError());
        QCK(hipStreamSynchronize(s));
        memcpy(hits, B->out[0], n64 * sizeof(stc_hit));
        *done = true;
        return STC_OK;
    }
    uint64_t *ka = (uint64_t *)B->sort, *kb2 = ka + n;
    uint32_t *va = (uint32_t *)(kb2 + n), *vb = va + n, *temp = vb + n;
    *B->wide = 0;
    bool alt = false;
    hipLaunchKernelGGL(k_hit_keys, dim3(blocks(n, 256)), dim3(256), 0, s, B->hits, (const uint32_t *)nullptr, n, kb, 0, ka, B->wide);
    int rc = stc_radix_sort_u64(ka, nullptr, kb2, va, ka, vb, n, 0, (int)(kb.two ? lb : hb + lb), temp, &alt, s);
    if (rc) return rc;
    uint32_t *idx = alt ? vb : va;
    if (kb.two) {
        uint32_t *other = alt ? va : vb;
        hipLaunchKernelGGL(k_hit_keys, dim3(blocks(n, 256)), dim3(256), 0, s, B->hits, (const uint32_t *)idx, n, kb, 1, ka, B->wide);
        bool alt2 = false;
        rc = stc_radix_sort_u64(ka, idx, ka, idx, kb2, other, n, 0, (int)hb, temp, &alt2, s);
        if (rc) return rc;
        if (alt2) idx = other;
    }
    QCK(hipGetLastError());
    const uint32_t chunks = (n + QFETCH - 1) / QFETCH;
    auto gather = [&](uint32_t c) {
        const uint32_t first = c * QFETCH, words = std::min(QFETCH, n - first) * 7;
        hipLaunchKernelGGL(k_hit_gather, dim3(blocks(words, 256)), dim3(256), 0, s, (const uint64_t *)B->hits, (const uint32_t *)idx,
                           first, words, (uint64_t *)B->out[c & 1]);
        return hipEventRecord(B->out_ev[c & 1], s);
    };
    QCK(gather(0));
    for (uint32_t c = 0; c < chunks; c++) {
        if (c + 1 < chunks) QCK(gather(c + 1));
        QCK(hipEventSynchronize(B->out_ev[c & 1]));
        if (*(volatile uint32_t *)B->wide) { /* let the gather in flight end before its buffer is used again */
            QCK(hipStreamSynchronize(s));
            return STC_OK;
        }
        const uint64_t first = (uint64_t)c * QFETCH;
        memcpy(hits + first, B->out[c & 1], std::min<uint64_t>(QFETCH, n - first) * sizeof(stc_hit));
    }
    *done = true;
    return STC_OK;
}

/* the decoded boxes of a CTF lie in [low, low + |extent| + longer edge] per
 * axis (new_parse_mbr): a conservative test, widened by 1e-6 degrees for the
 * float/double rounding of the bounds */
static bool ctf_may_intersect(const stc_ctf_meta &c, const double *box) {
    const double w0 = (double)(c.mbr[2] - c.mbr[0]), w1 = (double)(c.mbr[3] - c.mbr[1]);
    const double L = std::max(std::fabs(w0), std::fabs(w1)), eps = 1e-6;
    const double lo0 = (double)c.mbr[0] - std::fabs(w0) - eps, hi0 = (double)c.mbr[0] + std::fabs(w0) + L + eps;
    const double lo1 = (double)c.mbr[1] - std::fabs(w1) - eps, hi1 = (double)c.mbr[1] + std::fabs(w1) + L + eps;
    if (!(lo0 == lo0 && hi0 == hi0 && lo1 == lo1 && hi1 == hi1)) return true; /* NaN bounds: scan */
    return box[0] <= hi0 && box[2] >= lo0 && box[1] <= hi1 && box[3] >= lo1;
}

/* The tables of a batch that its kernels look into, and their bytes on the device (from the counts alone, before the
 * longest of them, the cells' lists, is made). */
struct QueryTables {
    std::vector<uint32_t> oq, rq;            /* object and pair queries, range queries */
    uint32_t bits = 0, f_bits = 5;           /* of the id hash; of the scans' id filter */
    std::vector<uint32_t> key;               /* hash of the queried ids */
    std::vector<int32_t> head, next;
    std::vector<uint32_t> start, list;       /* range queries by grid cell */
    std::vector<uint32_t> filter;
    uint64_t listed = 0, bytes = 0;

    template <class F>
    static void cells(const stc_query &q, const double *map, F f) {
        const double ix = QGRID / (map[2] - map[0]), iy = QGRID / (map[3] - map[1]);
        const double *b = q.box;
        const int cx0 = grid_cell(b[0], map[0], ix), cx1 = grid_cell(b[2], map[0], ix);
        const int cy0 = grid_cell(b[1], map[1], iy), cy1 = grid_cell(b[3], map[1], iy);
        for (int cy = cy0; cy <= cy1; cy++)
            for (int cx = cx0; cx <= cx1; cx++) f(cy * QGRID + cx);
    }

    void plan(const stc_query *q, uint32_t nq, const double *map) {
        for (uint32_t i = 0; i < nq; i++) (q[i].kind == STC_Q_RANGE ? rq : oq).push_back(i);
        if (!oq.empty()) {
            bits = 6;
            while ((1ull << bits) < 2ull * oq.size()) bits++;
            const uint32_t size = 1u << bits, mask = size - 1;
            key.assign(size, 0xFFFFFFFFu);
            head.assign(size, -1);
            next.assign(nq, -1);
            for (size_t j = oq.size(); j-- > 0;) { /* insert in reverse: lists keep query order */
                uint32_t qi = oq[j], id = q[qi].oid, h = oid_slot(id, bits);
                while (key[h] != 0xFFFFFFFFu && key[h] != id) h = (h + 1) & mask;
                key[h] = id;
                next[qi] = head[h];
                head[h] = (int32_t)qi;
            }
            /* the scans' filter: 64 bits or more per queried id, 2^16 (8 KB of LDS) at most */
            f_bits = std::min(bits + 5, 16u);
        }
        filter.assign((1u << f_bits) / 32 + QGRID * QGRID / 32 + (rq.empty() ? 0 : QFINE * QFINE / 32), 0u);
        for (uint32_t i : oq) {
            const uint32_t h = oid_slot(q[i].oid, f_bits);
            filter[h >> 5] |= 1u << (h & 31);
        }
        if (!rq.empty()) { /* counted per cell; listed in query order by list_cells */
            uint32_t *cell_bits = filter.data() + (1u << f_bits) / 32;
            start.assign(QGRID * QGRID + 1, 0);
            for (uint32_t qi : rq) cells(q[qi], map, [&](int c) { start[c + 1]++; });
            for (int c = 0; c < QGRID * QGRID; c++) {
                listed += start[c + 1];
                if (start[c + 1]) cell_bits[c >> 5] |= 1u << (c & 31);
                start[c + 1] = (uint32_t)listed;
            }
            /* the fine grid's cells at and around the boxes; all of them where the map is too small for 32 bits */
            const double x0 = map[0], y0 = map[1], ix = QGRID / (map[2] - map[0]), iy = QGRID / (map[3] - map[1]);
            uint32_t *fine = cell_bits + QGRID * QGRID / 32;
            const double fine_per = (double)QFINE / QGRID;
            auto fine_of = [&](double v, double v0, double inv, int off) {
                const double f = (v - v0) * inv * fine_per;
                return std::min(std::max((!(f >= 0.0) ? 0 : f >= (double)QFINE ? QFINE - 1 : (int)f) + off, 0), QFINE - 1);
            };
            if (!(ix < 1e30 && iy < 1e30)) std::fill(fine, fine + QFINE * QFINE / 32, ~0u);
            else
                for (uint32_t qi : rq) {
                    const double *b = q[qi].box;
                    const int x0c = fine_of(b[0], x0, ix, -1), x1c = fine_of(b[2], x0, ix, 1);
                    for (int y = fine_of(b[1], y0, iy, -1); y <= fine_of(b[3], y0, iy, 1); y++)
                        for (int w = x0c >> 5; w <= x1c >> 5; w++)
                            fine[y * (QFINE / 32) + w] |= (w == x0c >> 5 ? ~0u << (x0c & 31) : ~0u) & (w == x1c >> 5 ? ~0u >> (31 - (x1c & 31)) : ~0u);
                }
        }
        for (uint64_t b : std::initializer_list<uint64_t>{(nq + 1ull) * 8, nq * sizeof(stc_query), key.size() * 4ull, head.size() * 4ull,
                                                          next.size() * 4ull, oq.size() * 4ull, start.size() * 4ull, listed * 4, filter.size() * 4ull})
            bytes += QueryUpload::room(b);
    }

    void list_cells(const stc_query *q, const double *map) {
        if (rq.empty()) return;
        list.resize(listed);
        std::vector<uint32_t> at(start.begin(), start.end() - 1);
        for (uint32_t qi : rq) cells(q[qi], map, [&](int c) { list[at[c]++] = qi; });
    }
};

uint64_t stc_query_table_bytes(const stc_query *q, uint32_t nq, const double *map) {
    QueryTables t;
    t.plan(q, nq, map);
    return t.bytes;
}

/* device memory for `need` bytes more, with the reserve left? */
bool QueryAdmission::fits(uint64_t more) {
    size_t total_b = 0, free_b = 0;
    if (!more || hipMemGetInfo(&free_b, &total_b) != hipSuccess) return true;
    free = free_b;
    return more + reserve <= free_b;
}
int QueryAdmission::refuse(uint64_t more) {
    need = more;
    refused = true;
    return STC_E_CAPACITY;
}

int stc_query_run(QueryBufs *B, const QueryState &st, const stc_query *q, uint32_t nq, stc_hit *hits, uint64_t cap,
                  uint64_t *n_hits, uint64_t *counts, QueryAdmission &adm, QueryRoom *more, hipStream_t s) {
    if (nq == 0) {
        *n_hits = 0;
        if (more) more->all = true;
        return STC_OK;
    }
    QueryTables T;
    T.plan(q, nq, st.map);
    const std::vector<uint32_t> &oq = T.oq, &rq = T.rq;
    const uint32_t nruns = (uint32_t)st.runs.size();
    const uint64_t hits_need = std::max<uint64_t>(hits ? cap : 0, 1);
    const uint64_t need = B->batch.growth(T.bytes) + (hits_need > B->hits_cap ? hits_need * sizeof(stc_hit) * 3 / 2 : 0);
    if (T.listed > 0xFFFFFFFFull || !adm.fits(need)) return adm.refuse(need);
    T.list_cells(q, st.map);
    const uint64_t bytes = T.bytes;
    const uint64_t most = hits ? std::min<uint64_t>(cap, QSORT_HOST) : 0, res_words = nq + 1ull + most * 7;
    if (B->batch.begin(bytes) || grow(&B->hits, &B->hits_cap, hits_need))
        return stc_hip_fail(hipErrorOutOfMemory, "query buffers", __FILE__, __LINE__);
    if (B->res_cap < res_words) {
        B->free_res();
        if (hipHostMalloc((void **)&B->res, (res_words + res_words / 2) * 8, hipHostMallocDefault) == hipSuccess) {
            B->res_cap = res_words + res_words / 2;
        } else { /* the counters are copied instead, and the hits with them */
            B->res = nullptr;
            (void)hipGetLastError();
        }
    }
    QueryUpload &U = B->batch;
    QDev Q;
    unsigned long long *counters = U.put((const unsigned long long *)nullptr, nq + 1ull); /* total hits, then per query */
    Q.q = U.put(q, nq);
    Q.oh_key = U.put(T.key.data(), T.key.size());
    Q.oh_head = U.put(T.head.data(), T.head.size());
    Q.q_next = U.put(T.next.data(), T.next.size());
    const uint32_t *oq_dev = U.put(oq.data(), oq.size());
    Q.g_start = U.put(T.start.data(), T.start.size());
    Q.g_list = U.put(T.list.data(), T.list.size());
    Q.filter = U.put(T.filter.data(), T.filter.size());
    Q.f_bits = T.f_bits;
    Q.oh_bits = T.bits;
    Q.n_range = (uint32_t)rq.size();
    const double x0 = st.map[0], y0 = st.map[1];
    const double ix = QGRID / (st.map[2] - st.map[0]), iy = QGRID / (st.map[3] - st.map[1]);
    Q.x0 = x0;
    Q.y0 = y0;
    Q.ix = ix;
    Q.iy = iy;
    Q.fx[0] = (float)x0;
    Q.fx[1] = (float)(x0 - (double)Q.fx[0]);
    Q.fy[0] = (float)y0;
    Q.fy[1] = (float)(y0 - (double)Q.fy[0]);
    Q.fix = (float)(ix * (QFINE / QGRID));
    Q.fiy = (float)(iy * (QFINE / QGRID));
    Q.hits = B->hits;
    Q.cap = more ? B->hits_cap : hits ? cap : 0;
    Q.n_hits = counters;
    Q.counts = counters + 1;
    Q.nq = nq;
    Q.lds = nq <= QLDS;
    const size_t q_scan_lds = ((Q.lds ? nq : 0) + T.filter.size()) * sizeof(uint32_t);
    QCK(U.send(s));
    /* counts a planner adds without a kernel (CTFs wholly inside a range query) */
    std::vector<unsigned long long> planned(nq, 0);

    /* live meetings and memtable */
    if (st.stepped && st.meets.base && st.nb) {
        const dim3 g((uint32_t)std::min<uint64_t>(blocks(st.nb, 256), 4096));
        bool stores = false;
        for (uint32_t i = 0; i < nq && Q.cap && !stores; i++) stores = !(q[i].flags & STC_QF_COUNT);
#define Q_LIVE(OIDS, RANGES)                                                                                                        \
    do {                                                                                                                            \
        if (stores) hipLaunchKernelGGL((k_q_live<OIDS, RANGES, true>), g, dim3(256), q_scan_lds, s, st.meets, st.nb, st.last_t, Q); \
        else hipLaunchKernelGGL((k_q_live<OIDS, RANGES, false>), g, dim3(256), q_scan_lds, s, st.meets, st.nb, st.last_t, Q);       \
    } while (0)
        if (Q.n_range && T.bits) Q_LIVE(true, true);
        else if (Q.n_range) Q_LIVE(false, true);
        else if (T.bits) Q_LIVE(true, false);
#undef Q_LIVE
        QCK(hipGetLastError());
    }
    if (st.n_rec) {
        hipLaunchKernelGGL(k_q_mem, dim3(std::min<uint32_t>(blocks(st.n_rec, 256), 4096)), dim3(256), q_scan_lds, s,
                           st.rec_keys, st.rec_boxes, st.n_rec, st.end_time_min, Q);
        QCK(hipGetLastError());
    }
    /* runs */
    if (nruns) {
        std::vector<uint4> cand;
        if (!rq.empty()) { /* while the scans run */
            for (uint32_t qi : rq) {
                const stc_query &qq = q[qi];
                for (uint32_t r = 0; r < nruns; r++) {
                    const stc_ctf_meta *ctfs = st.run_ctfs[r];
                    const CtfStats *cs = st.run_stats[r];
                    for (uint32_t c = 0; c < st.runs[r].ctf_count; c++) {
                        if (!ctfs[c].kv_capacity) continue;
                        if (cs && cs[c].regular) {
                            const CtfStats &x = cs[c];
                            /* no record can match */
                            if (!(x.box[0] <= qq.box[2] && x.box[2] >= qq.box[0] && x.box[1] <= qq.box[3] &&
                                  x.box[3] >= qq.box[1]) || x.start_min > qq.t1 || x.end_max < qq.t0)
                                continue;
                            /* every forward record matches: count without decoding */
                            if ((!Q.cap || (qq.flags & STC_QF_COUNT)) && x.box[0] >= qq.box[0] &&
                                x.box[2] <= qq.box[2] && x.box[1] >= qq.box[1] &&
                                x.box[3] <= qq.box[3] && x.start_min >= qq.t0 && x.end_max <= qq.t1) {
                                planned[qi] += x.n_fwd;
                                continue;
                            }
                        } else if (!ctf_may_intersect(ctfs[c], qq.box)) {
                            continue;
                        }
                        cand.push_back(make_uint4(qi, r, c, 0));
                    }
                    if (st.runs[r].n_tail) cand.push_back(make_uint4(qi, r, 0xFFFFFFFFu, 0));
                }
            }
        }
        if (!oq.empty() || !cand.empty()) {
            /* their number is known while the scans run: planned ahead of them, a batch of 2,000 would wait for the plan */
            const uint64_t rb = QueryUpload::room(nruns * sizeof(QueryRunDev)) + QueryUpload::room(cand.size() * sizeof(uint4)),
                           growth = B->runs.growth(rb);
            if (!adm.fits(growth)) {
                QCK(hipStreamSynchronize(s)); /* the scans, which read the batch's tables */
                return adm.refuse(growth);
            }
            if (B->runs.begin(rb)) {
                (void)hipStreamSynchronize(s);
                return stc_hip_fail(hipErrorOutOfMemory, "query runs", __FILE__, __LINE__);
            }
            const QueryRunDev *runs = B->runs.put(st.runs.data(), nruns);
            const uint4 *cand_dev = B->runs.put(cand.data(), cand.size());
            QCK(B->runs.send(s));
            if (!oq.empty())
                hipLaunchKernelGGL(k_q_run_oid, dim3(blocks((uint64_t)oq.size() * nruns * STC_WAVE, 256)), dim3(256), 0, s, runs,
                                   nruns, oq_dev, (uint32_t)oq.size(), st.num_objects, Q);
            QCK(hipGetLastError());
            if (!cand.empty())
                hipLaunchKernelGGL(k_q_run_range, dim3((uint32_t)cand.size()), dim3(256), 0, s, runs, cand_dev, Q);
            QCK(hipGetLastError());
        }
    }

    /* results */
    std::vector<uint64_t> copied;
    if (B->res) {
        hipLaunchKernelGGL(k_q_finish, dim3(std::min<uint32_t>(blocks(res_words, 256), 256)), dim3(256), 0, s, counters, nq,
                           (const uint64_t *)B->hits, most, B->res);
        QCK(hipGetLastError());
    } else {
        copied.resize(nq + 1ull);
        QCK(hipMemcpyAsync(copied.data(), counters, (nq + 1ull) * 8, hipMemcpyDeviceToHost, s));
    }
    QCK(hipStreamSynchronize(s));
    const uint64_t *cnt = B->res ? B->res : copied.data();
    uint64_t total = 0; /* the hits of the queries that store theirs */
    for (uint32_t i = 0; i < nq; i++) {
        const uint64_t ci = cnt[i + 1] + planned[i];
        if (!(q[i].flags & STC_QF_COUNT)) total += ci;
        if (counts) counts[i] = ci;
    }
    *n_hits = total;
    if (more) {
        more->all = total <= Q.cap;
        if (more->all && total > cap) {
            stc_hit *all = more->room(more->arg, total);
            more->all = all != nullptr;
            hits = all;
            cap = total;
        }
        if (!more->all) return STC_OK;
    }
    uint64_t stored = Q.cap ? std::min<uint64_t>(cnt[0], cap) : 0;
    bool sorted = false;
    if (stored > QSORT_HOST && hits) {
        const int rc = fetch_sorted(B, st, nq, stored, hits, adm.reserve, &sorted, s);
        if (rc) return rc;
    }
    if (stored && hits && !sorted) {
        if (B->res && stored <= most) memcpy(hits, cnt + nq + 1, stored * sizeof(stc_hit));
        else QCK(hipMemcpy(hits, B->hits, stored * sizeof(stc_hit), hipMemcpyDeviceToHost));
        std::sort(hits, hits + stored, [](const stc_hit &a, const stc_hit &b) {
            if (a.query != b.query) return a.query < b.query;
            if (a.source != b.source) return a.source < b.source;
            if (a.pid != b.pid) return a.pid < b.pid;
            if (a.target != b.target) return a.target < b.target;
            if (a.start != b.start) return a.start < b.start;
            return a.end < b.end;
        });
    }
    return STC_OK;
}
