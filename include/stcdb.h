/*
 * stcdb.h — C ABI of the MI355X co-occurrence pipeline (libstcdb_hip.so).
 *
 * This is the drop-in boundary for the reference's GPU path. The reference
 * selects its GPU path at compile time (USE_GPU, src/Makefile:28-32) and
 * binds three C++ functions:
 *
 *   vector<gpu_info*> get_gpus()                                src/cuda/cuda_common.cu:48
 *   workbench *cuda_create_device_bench(workbench*, gpu_info*)  src/cuda/geometry.cu:1395
 *   void process_with_gpu(workbench*, workbench*, gpu_info*)    src/cuda/geometry.cu:1573
 *     (declared at src/tracing/process.cpp:373-376, called at :423 and :462)
 *
 * They pass whole workbench structs by pointer and exit() on any CUDA error
 * (CUDA_SAFE_CALL, src/cuda/cuda_util.cuh:19-27). Here the same operations
 * take plain structs, pointers and sizes, return status codes, and keep all
 * device state behind an opaque context. All functions are thread-compatible:
 * one context per host thread.
 *
 * Status codes: STC_OK (0) or a negative STC_E_* value; stc_last_error()
 * gives the message of the last failure on a context.
 */
#ifndef STCDB_H_
#define STCDB_H_

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define STC_OK 0
#define STC_E_ARG (-1)       /* invalid argument or configuration */
#define STC_E_HIP (-2)       /* HIP runtime error (no device, launch failure, ...) */
#define STC_E_CAPACITY (-3)  /* a device buffer would overflow and could not grow */
#define STC_E_INPUT (-4)     /* a point lies outside the map box */
#define STC_E_STATE (-5)     /* call out of order (e.g. inspection before any step) */

/* compat bits */
#define STC_COMPAT_HALF_REDUCTION 1u /* reproduce geometry.cu:865-888 and 955-974 */

/* Configuration: the subset of the reference's `configuration`
 * (src/util/config.h:15-86) that the GPU path reads. */
typedef struct stc_config {
    uint32_t num_objects;         /* config->num_objects */
    uint32_t grid_capacity;       /* config->grid_capacity: a QTree block splits above it */
    double grid_amplify;          /* config->grid_amplify: points stored per leaf = amplify * capacity */
    uint32_t min_meet_time;       /* config->min_meet_time (seconds) */
    uint32_t max_meet_time;       /* config->max_meet_time (seconds); longer meetings go to the oversize buffer */
    uint32_t start_time;          /* config->start_time */
    uint32_t kv_restriction;      /* flush once the memtable holds more records (config->kv_restriction) */
    uint32_t ctf_count;           /* config->CTF_count, a square */
    uint32_t compat;              /* STC_COMPAT_* bits */
    uint64_t num_meeting_buckets; /* initial meeting-array size; 0 = 2 * num_objects (config.h:306-308). Grows on demand. */
    double reach_distance;        /* config->reach_distance (metres) */
    double area_threshold;        /* workbench::dProbFalse: object MBR area (deg^2) above which it is oversize */
    uint32_t keep_pairs;          /* bit 0: keep each step's pair list for stc_get_pairs;
                                     bit 1: keep each run's sorted records for stc_get_run */
    uint32_t device_runs;         /* nonzero: keep every flushed run in HBM for stc_query until stc_drop_runs */
    uint32_t dynamic_schema;      /* config->dynamic_schema (config.h:35, the reference's default).
                                     Nonzero: one QTree kept across steps, built from the first
                                     step's points as partitioner::build_schema builds it
                                     (filter.cpp:27-93) or installed with stc_set_schema, and
                                     split/merged after every step (geometry.cu:1114-1234, 2159-2182).
                                     Zero: the QTree is rebuilt from every step's points
                                     (--disable_dynamic_schema, geometry.cu:1629-1651). */
    uint32_t schema_update_delay; /* config->schema_update_delay (config.h:38); 0 counts as 1 */
    uint32_t async_flush;         /* nonzero: a step's flush runs on its own stream from a host thread
                                     and overlaps the next step up to that step's merge, which reuses
                                     the memtable. The run is the same; every call that reads runs
                                     (stc_num_runs, stc_get_run_info, stc_get_run, stc_dump_run,
                                     stc_drop_runs, stc_compact_runs, stc_sync, stc_get_records)
                                     waits for it, and query batches see the state before the flush
                                     until then. Zero: the flush completes inside the step
                                     (process_with_gpu's order). */
} stc_config;

/* A QTree node: the reference's QTSchema (src/index/QTree.h:49-62), 80 bytes,
 * as create_schema flattens a QTNode tree (QTree.h:286-311): node 0 is the
 * root, a branch's children are node indices in the order bottom-left,
 * bottom-right, top-left, top-right (QTree.h:24-29). */
typedef struct stc_qtnode {
    uint32_t grid_id;          /* a leaf's grid (ignored by stc_set_schema: leaves are renumbered) */
    int16_t level;
    int16_t type;              /* 0 invalid (a free slot), 1 BRANCH, 2 LEAF */
    int16_t overflow_count, underflow_count;
    double mid_x, mid_y;
    double mbr[4];             /* low0, low1, high0, high1 */
    uint32_t children[4];
} stc_qtnode;

typedef struct stc_box {
    double low[2];
    double high[2];
} stc_box;

/* Per-step counters, the fields process_with_gpu copies back to the host
 * workbench (geometry.cu:1655-1745) plus device-side stage timings. */
typedef struct stc_step_out {
    uint64_t nodes;            /* QTree nodes built this step */
    uint64_t leaves;           /* QTree leaves (grids) */
    uint64_t border_points;    /* filter_list_index */
    uint64_t cross_units;      /* point-leaf checks added by the border lookup */
    uint64_t candidates;       /* point pairs whose distance was evaluated */
    uint64_t pairs;            /* unique pairs within reach_distance */
    uint64_t active_meetings;  /* num_active_meetings */
    uint64_t expired;          /* meetings that ended this step (emitted or not) */
    uint64_t new_records;      /* records added to the memtable this step */
    uint64_t kv_count;         /* records in the memtable after the step (before a flush) */
    uint64_t overflow_points;  /* points beyond the leaf buffer (not stored as targets) */
    uint64_t ambiguous_pairs;  /* pair decisions re-evaluated on the host (distance within 16 ulp of r) */
    uint64_t ambiguous_nodes;  /* box-distance decisions within 16 ulp of r (decided on the device) */
    uint64_t table_buckets;    /* buckets of this step's meeting array: live meetings and dead slots */
    uint64_t table_occupied;   /* num_taken_buckets: meetings held when identify ran (active + expired) */
    uint32_t flushed;          /* 1 if this step flushed a run */
    uint32_t rebuilt;          /* 0 (every step's merge writes a new meeting array) */
    float ms_partition;        /* QTree build + partition */
    float ms_filter;           /* border lookup */
    float ms_refine;           /* pair refinement: reverse lists, collect, place, segment sorts */
    float ms_meetings;         /* merge with the previous meetings + records */
    float ms_flush;            /* flush (0 when no flush) */
    float ms_total;
    float ms_refine_kernel;    /* the pair place pass (owner segments, sorted) */
    float ms_identify_kernel;  /* the merge with the previous meetings (last launch) */
    uint64_t continuing;       /* pairs that continued a meeting of the previous step */
    uint64_t new_keys;         /* pairs that opened a meeting */
    float ms_count_kernel;     /* the pair collect pass (last launch) */
    float ms_schema;           /* dynamic schema update after the step (pro.index_update_time) */
    float ms_flush_done;       /* device time of the flush that completed during this call: this
                                  step's (= ms_flush), or with async_flush the previous step's */
} stc_step_out;

/* CTF metadata of a flushed run: the fields of the reference's CTF
 * (src/tracing/step_merge.h:64-109) without its host pointers. */
typedef struct stc_ctf_meta {
    float mbr[4];              /* ctf_mbr: low0, low1, high0, high1 */
    uint32_t kv_capacity;
    uint32_t start_time_min, start_time_max;
    uint32_t end_time_min, end_time_max;
    uint32_t bitmap_size;      /* bytes of the bitmap written with the CTF meta */
    uint16_t key_bit, id_bit, duration_bit, end_bit;
    uint16_t low_x_bit, low_y_bit, edge_bit, mbr_bit;
    uint16_t x_grid, y_grid;
    uint32_t flags;            /* bit0: the reference would fail an assert on this CTF */
} stc_ctf_meta;

/* A flushed run (the reference's CTB, src/tracing/step_merge.h:111-131, and
 * its oversize buffer, :44-62). */
typedef struct stc_run_info {
    uint32_t kv_count;         /* records stored in the CTFs */
    uint32_t oversize_count;   /* records in the oversize buffer */
    uint32_t ctf_count;
    uint32_t num_objects;
    uint32_t o_start_min, o_start_max, o_end_min, o_end_max; /* oversize buffer time bounds */
    uint32_t end_time_min;     /* time base of the end offsets in this run's keys */
    uint32_t cur_time;         /* timestep that triggered the flush */
    uint32_t sid_count, oversize_oid_count;
    uint64_t key_bytes;        /* packed CTF key bytes over all CTFs */
} stc_run_info;

/* Device description (the reference's gpu_info, src/cuda/mygpu.h:18-50). */
typedef struct stc_device_info {
    int32_t device_id;
    char name[256];
    uint64_t mem_size;
    int32_t num_cus;
    int32_t clock_khz;
} stc_device_info;

/* ---- device discovery: replaces get_gpus() (cuda_common.cu:48-72) ---- */
int stc_device_count(int32_t *count);
int stc_device_info_get(int32_t device, stc_device_info *info);

/* ---- lifecycle: replaces cuda_create_device_bench (geometry.cu:1395-1565) ----
 * Allocates all device state for `cfg` on the current HIP device. map_mbr is
 * the map box (tracer::mbr). */
int stc_create(const stc_config *cfg, const stc_box *map_mbr, void **ctx);

/* ---- dynamic schema (cfg.dynamic_schema) ----
 * stc_build_schema builds the initial QTree from one timestep's num_objects
 * AoS points (host memory, or device memory when xy_on_device) as
 * partitioner::build_schema does (filter.cpp:27-93 with QTNode::insert/split,
 * QTree.h:157-214): a node splits when at least grid_capacity points reach it
 * and half its width in metres at its low latitude exceeds reach_distance;
 * children are the exact halves of its box. The build runs on the device.
 * Without it, the first stc_step builds the tree from its own points (the
 * reference builds it from the first timestep, process.cpp:401-402).
 * stc_set_schema installs a tree the host built instead (bench->schema, which
 * cuda_create_device_bench copies to the device, geometry.cu:1395-1565); it is
 * checked to be a tree over the map box with leaves and branches only below
 * node 0, and STC_E_ARG is returned otherwise. stc_get_schema copies the
 * current tree out (after a step: the tree the next step will use); grid_id
 * of a leaf is its leaf number in stc_get_leaves order of slots. All three
 * return STC_E_STATE when the context rebuilds its tree every step. */
int stc_build_schema(void *ctx, const double *xy, int32_t xy_on_device);
int stc_set_schema(void *ctx, const stc_qtnode *nodes, uint32_t n_nodes);
int stc_get_schema(void *ctx, stc_qtnode *nodes, uint64_t cap, uint64_t *n);
int stc_destroy(void *ctx);
const char *stc_last_error(void *ctx);

/* ---- one timestep: replaces process_with_gpu (geometry.cu:1573-2218) ----
 * xy: num_objects AoS (x, y) doubles in degrees (the reference's Point array,
 * geometry.h:23-56). stc_step copies host memory to the device first;
 * stc_step_device takes a device pointer already resident in HBM. t is
 * bench->cur_time. A flush runs inside the step when the memtable exceeds
 * kv_restriction, as in process_with_gpu; its run is then available through
 * stc_num_runs/stc_get_run. */
int stc_step(void *ctx, const double *xy_host, uint32_t t, stc_step_out *out);
int stc_step_device(void *ctx, const double *xy_dev, uint32_t t, stc_step_out *out);

/* ---- batched streams ----
 * One timestep of n independent contexts (the reference's batched streams,
 * one context each): every context steps as stc_step (xy[i] in host memory)
 * or stc_step_device (on_device[i] nonzero; on_device may be null) would, on
 * its own streams, driven from up to `threads` host threads (largest contexts
 * first) so that their kernels overlap on the device. outs[i] and rcs[i]
 * (either may be null) receive context i's counters and status. Returns
 * STC_OK when every step succeeded, else the first failing context's code,
 * its message in that context's stc_last_error. Contexts must be distinct and
 * must not be in use by other threads during the call. Each context's result
 * equals its own sequential run. No counterpart in the reference, which runs
 * one stream per process invocation. */
int stc_step_batch(void *const *ctxs, uint32_t n, const double *const *xy, const int32_t *on_device, uint32_t t,
                   uint32_t threads, stc_step_out *outs, int32_t *rcs);

/* ---- per-second meeting persistence ----
 * The reference can save the pairs each step finds and replay them later in
 * place of the positions (save_meetings_pers / load_meetings_pers:
 * geometry.cu:456-466, 1609-1622, 1718-1723; files by workbench::dump_meetings
 * and load_meetings, workbench.cpp:446-470). One unit per pair and step, the
 * reference's 32-byte meeting_unit (workbench.h:62-83). */
typedef struct stc_meeting_unit {
    uint64_t key;              /* Cantor key of (min pid, max pid): (a + b)(a + b + 1)/2 + b */
    uint32_t start, end;       /* the step (a replay ignores them, as insert_meetings_to_buckets does) */
    float mbr[4];              /* float bbox of the two positions at the step: low0, low1, high0, high1 */
} stc_meeting_unit;

/* the last step's pairs as units, in pair order; needs keep_pairs bit 0 */
int stc_get_step_meetings(void *ctx, stc_meeting_unit *units, uint64_t cap, uint64_t *n);
/* A step from units instead of positions (insert_meetings_to_buckets,
 * geometry.cu:544-565, without its 5-probe drop): each pair is inserted or
 * extended with its MBR, then meetings are identified and the memtable
 * flushed as in stc_step. Each pair at most once per call (STC_E_INPUT
 * otherwise, and for keys naming no two distinct objects below num_objects);
 * fewer than 2^32 - 1 units. No tree is built, so the step reports no nodes,
 * leaves or candidates. */
int stc_step_meetings(void *ctx, const stc_meeting_unit *units, uint64_t n, uint32_t t, stc_step_out *out);

/* ---- inspection of the current state (copies to host memory) ----
 * Each getter writes at most `cap` items and stores the total count in *n. */
int stc_get_pairs(void *ctx, uint64_t *keys, uint64_t cap, uint64_t *n);   /* last step, sorted, oid1<<32|oid2 */
int stc_get_active(void *ctx, uint64_t *keys, uint32_t *start, uint32_t *end, float *mbr, uint64_t cap, uint64_t *n);
int stc_get_records(void *ctx, uint64_t *keys, float *boxes, uint64_t cap, uint64_t *n); /* memtable, keys as lo,hi */
int stc_get_leaves(void *ctx, double *boxes, uint32_t *counts, uint64_t cap, uint64_t *n); /* last step's leaves */

/* ---- flushed runs ---- */
int stc_num_runs(void *ctx, uint32_t *n);
int stc_get_run_info(void *ctx, uint32_t run, stc_run_info *info);
/* any output pointer may be NULL; sizes follow stc_run_info:
 * ctfs[ctf_count], key_bytes[key_bytes], bitmaps[ctf_count * 8192],
 * sids[num_objects], o_keys[2 * oversize_count], o_boxes[4 * oversize_count],
 * o_bitmap[8192], sorted_keys[2 * kv_count], sorted_boxes[4 * kv_count] */
int stc_get_run(void *ctx, uint32_t run, stc_ctf_meta *ctfs, uint8_t *key_bytes, uint8_t *bitmaps,
                uint16_t *sids, uint64_t *o_keys, float *o_boxes, uint8_t *o_bitmap,
                uint64_t *sorted_keys, float *sorted_boxes);
int stc_drop_runs(void *ctx); /* release host copies of flushed runs (owed copies still complete); with an
                                 asynchronous flush in progress the release happens when it joins, its run
                                 included */
/* CTF::get_ctf_bits (src/tracing/step_merge.cpp:140-186), which the
 * reference's host runs for every CTF of a flush (geometry.cu:1960-1964):
 * fills the id, duration, end, low_x, low_y, edge and mbr bit widths, key_bit,
 * the bitmap grid (x_grid, y_grid) and bitmap_size of `ctf` from its mbr (set
 * by the caller), the map box, the object count and max_meet_time. flags bit 0
 * is set where the reference would fail an assert. Host arithmetic only; needs
 * no device. */
int stc_ctf_widths(stc_ctf_meta *ctf, const stc_box *map_mbr, uint32_t num_objects, uint32_t max_meet_time);
/* Compaction: merge runs [first, first + count) into one run that takes their
 * place (later runs move down by count - 1). The records of the inputs are
 * decoded as the reference's compaction reads them (CTF::parse_key and
 * CTF::new_parse_mbr_f_box, tools/compaction.cpp:320-336), their end times
 * re-based on the earliest input base (compaction.cpp:483-487), and flushed
 * again: STR partition, CTF encoding and bitmaps as in a step's flush, with
 * objects oversize in any input kept oversize (compaction.cpp:259-268). The
 * inputs must be kept in HBM (stc_config.device_runs). Replaces the offline
 * merge of tools/compaction.cpp:729-1206. */
int stc_compact_runs(void *ctx, uint32_t first, uint32_t count);
/* Wait until all work of the context is done, including the background copies
 * of flushed runs into host memory (a flush hands its run to a copy stream,
 * queued when the next step starts its pair count so that the copy overlaps
 * it; stc_get_run, stc_dump_run and stc_sync queue a waiting copy first, and
 * stc_get_run waits for its own run). */
int stc_sync(void *ctx);

/* ---- flushed runs on disk ----
 * Writes run `run` as the reference's straight_dump lays it out
 * (src/tracing/process.cpp:254-348): <dir>/<prefix>_SSTable_<ctb>-<c> (packed
 * keys of CTF c), <dir>/<prefix>_CTB<ctb> (the 128-byte CTB image, sids,
 * oversize keys, boxes and bitmap; workbench.cpp:597-614) and
 * <dir>/<prefix>_STcL<ctb>-<c> (the 80-byte CTF image and its bitmap;
 * step_merge.cpp:644-650). Pointer fields of the images are zero; CTB fields
 * the reference's GPU path leaves unset carry the run's CTF count, start-time
 * bounds, end-time base and flush time. */
int stc_dump_run(void *ctx, uint32_t run, const char *dir, const char *prefix, uint32_t ctb);

/* ---- queries over the resident state ----
 * The reference answers object-history, range and time queries from its
 * flushed runs (workbench::id_search_in_CTB, mbr_search_in_disk,
 * search_time_in_disk: src/tracing/workbench.cpp:350-572; CTF::search_SSTable,
 * time_search: src/tracing/step_merge.cpp:528-584). stc_query_batch answers a batch
 * over everything the context holds after the last step, with exact set
 * semantics:
 *   STC_Q_OID   meetings with pid == oid;
 *   STC_Q_RANGE meetings whose MBR intersects box (closed bounds, compared in
 *               double), each meeting once (the record with pid < target);
 *   STC_Q_PAIR  meetings with pid == oid and target == oid2;
 * each restricted to meetings whose [start, end] overlaps [t0, t1]. Sources:
 * live meetings (start, end = last step, f32 MBR; both directions), memtable
 * records (end = offset + time base, start = end - duration) and the runs kept
 * in HBM (device_runs), whose keys are decoded as CTF::ctf_get_key_oid,
 * parse_key and new_parse_mbr decode them (step_merge.cpp:325-379). counts[q]
 * is the number of hits of query q; at most `cap` hits are stored, sorted by
 * (query, source, pid, target, start, end), none of a query flagged
 * STC_QF_COUNT (the reference's box search counts, search_count at
 * workbench.cpp:478-572); *n_hits is the number of hits of the queries not
 * flagged STC_QF_COUNT (all of which fit when cap >= *n_hits). */
#define STC_Q_OID 1u
#define STC_Q_RANGE 2u
#define STC_Q_PAIR 3u

#define STC_QF_COUNT 1u     /* count the query's hits and store none (the reference's
                              * search_count; a range query can meet millions of records) */

typedef struct stc_query {
    uint32_t kind;
    uint32_t oid, oid2;
    uint32_t t0, t1;           /* inclusive time window */
    uint32_t flags;            /* STC_QF_* bits */
    double box[4];             /* STC_Q_RANGE: low0, low1, high0, high1 (degrees) */
} stc_query;

typedef struct stc_hit {
    uint32_t query;            /* index of the query in the batch */
    uint32_t pid, target;      /* the meeting as seen from pid */
    uint32_t start, end;
    uint32_t source;           /* 0 live, 1 memtable, 2 + r run r (stc_get_run numbering) */
    double mbr[4];             /* f32 MBR (live, memtable) or the decoded CTF MBR (runs) */
} stc_hit;

int stc_query_batch(void *ctx, const stc_query *q, uint32_t nq, stc_hit *hits, uint64_t cap, uint64_t *n_hits,
              uint64_t *counts);
/* The same for a caller that wants every hit and does not know how many there
 * are: up to cap go to hits; of more, room(arg, n) is asked for an array of
 * n, which takes them all, where the context's own hit buffer (as long as the
 * largest cap so far, and half again) held them. Where it did not, or room
 * gave null, *n_hits > cap and *all = 0: nothing is stored, and the batch is
 * asked again with cap = *n_hits. room is called on the calling thread, at
 * most once, and must not call into the context. */
typedef stc_hit *(*stc_room)(void *arg, uint64_t n);
int stc_query_batch_room(void *ctx, const stc_query *q, uint32_t nq, stc_hit *hits, uint64_t cap, stc_room room, void *arg,
              uint64_t *n_hits, uint64_t *counts, int32_t *all);
/* Serving. A query batch answers over the state the last completed step
 * published (its meetings, memtable and runs) and runs on the context's own
 * query stream, so batches issued from another host thread overlap the next
 * step on the device; that step waits only where it overwrites what an
 * earlier batch still reads (the other meeting array; the memtable from its
 * start after a flush). Batches are admitted by free device memory: one whose
 * tables (its queries, ids and the cells of its boxes), candidates and hit
 * buffer would leave less than 1 GiB free returns STC_E_CAPACITY (split it and
 * retry). stc_query_batch_at also reports the
 * timestep of the state it answered. Only stc_query_batch, stc_query_batch_room,
 * stc_query_batch_at and stc_live_search may run concurrently with stc_step on one context;
 * stc_drop_runs and stc_compact_runs wait for batches in flight. The
 * reference answers its live search from the command thread between steps
 * (process.cpp:350-371, 443-495). */
int stc_query_batch_at(void *ctx, const stc_query *q, uint32_t nq, stc_hit *hits, uint64_t cap, uint64_t *n_hits,
                       uint64_t *counts, uint32_t *state_step);

/* Live contact search (the reference's search_single / search_multi inside
 * cuda_identify_meetings, src/cuda/geometry.cu:605-662, driven from
 * src/tracing/process.cpp:465-495): the meetings live at the last step that
 * have lasted at least min_meet_time + 1 steps and involve one of `pids`, as
 * stc_hit records seen from the searched object (source 0). A second call
 * with the targets found is the reference's second hop. */
int stc_live_search(void *ctx, const uint32_t *pids, uint32_t n, stc_hit *hits, uint64_t cap, uint64_t *n_hits);

/* stc_live_search without allocation. This entry point has no counterpart in
 * the reference; it is for callers that cannot allocate (code under HIP graph
 * capture, tight serving loops, harnesses that forbid hipMalloc). Its results
 * are those of stc_live_search. Its scratch (the sorted search ids, a hit
 * counter and the staged hits) is one static device array of 14.8 MB per
 * device, set up by stc_create; on success the call makes no device or host
 * allocation. It reads the context's state directly: call it from the thread
 * that steps, not while a step runs. Limits: at most 16384 objects per call (STC_E_CAPACITY beyond)
 * and at most 262144 hits (STC_E_CAPACITY, *n_hits still set). Every call on
 * one GPU shares that GPU's array: calls that overlap on one GPU, from any
 * context or thread, race. */
int stc_live_search_noalloc(void *ctx, const uint32_t *pids, uint32_t n, stc_hit *hits, uint64_t cap,
                            uint64_t *n_hits);

/* ---- seeded synthetic traces (the reference's generator is unseeded) ----
 * Parameter and state layouts are those of stcdb_amd/csrc/stc_gen.h. */
typedef struct stc_gen_params stc_gen_params;
typedef struct stc_walker stc_walker;
int stc_gen_init_host(const stc_gen_params *p, stc_walker *w, uint32_t first, uint32_t count);
/* advance host walkers from step t-1 to t (t >= 1) */
int stc_gen_step_host(const stc_gen_params *p, stc_walker *w, uint32_t count, uint32_t t);
int stc_gen_pos_host(const stc_gen_params *p, const stc_walker *w, uint32_t count, double *xy);
/* device-resident trace: walkers live in HBM; stc_trace_next advances to t
 * (t == 0 returns the initial positions) and returns a device pointer to
 * num_objects AoS points valid until the next call. */
int stc_trace_create(const stc_gen_params *p, void **trace);
int stc_trace_next(void *trace, uint32_t t, const double **xy_dev);
int stc_trace_destroy(void *trace);

#ifdef __cplusplus
}
#endif
#endif /* STCDB_H_ */
