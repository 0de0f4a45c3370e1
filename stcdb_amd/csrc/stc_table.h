/*
 * stc_table.h — layout of the live meetings, shared by the pipeline and the
 * query kernels.
 *
 * A bucket is the reference's meeting_unit (src/tracing/workbench.h:62-83)
 * without its end time: 28 bytes of key, start and MBR. The MBR is stored as
 * order-preserving u32 images of the f32 bounds so that min/max updates are
 * integer ops. Keys are oid1 << 32 | oid2 with oid1 < oid2 < 2^26.
 *
 * The live meetings after a step are the buckets' keys, starts and MBRs, an
 * array each (a search by object then reads 8 bytes a meeting, not the lines
 * of all 28: a lookup among 10M meetings 52 -> 25 us; the merge, which reads
 * and writes all, takes 14.2 ms for 1.03e9 of either), sorted by key, one
 * segment per owner oid1 (a pair's smaller id). Bucket i of a step's array is
 * built from the step's pair slot i, so a slot that held a duplicate pair or
 * a rejected band pair leaves a dead bucket: key oid1 << 32 | DEAD_B (it sorts
 * after the owner's live pairs). The array has no free buckets: every bucket
 * is live or dead, and a live meeting was last seen at the step that built the
 * array, which is therefore its end time; the readers take it from the array's
 * step instead of from the bucket.
 */
#ifndef STC_TABLE_H_
#define STC_TABLE_H_

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>

#define DEAD_B 0xFFFFFFFFu /* partner word of a dead slot or bucket */

/* one meeting at hand */
struct __attribute__((packed, aligned(4))) Bucket {
    unsigned long long key;
    uint32_t start;
    uint32_t mbr[4];          /* ordered ints of low0, low1, high0, high1 */
};
static_assert(sizeof(Bucket) == 28, "a bucket is 28 bytes");

/* The three arrays of a step's meetings in one allocation, MBRs, keys, starts: each as long as the capacity, which is
 * a multiple of MEET_ROUND, so that each starts on a 4 KB boundary and every merge tile (128 meetings) begins and ends
 * on a line in all three. With a capacity of any length the keys and starts began at any multiple of 16 and 8 bytes,
 * and the merge's streaming stores shared lines between tiles: 1.03e9 meetings 13.8-15.7 ms into one of the two sets
 * and 14.8-16.7 into the other, over four pairs of runs on two boxes; 13.5-14.6 so (an allocation each: 13.6-14.6). */
#define MEET_ROUND 1024u
struct MeetLayout {
    size_t cap, keys, starts, bytes; /* meetings; where the keys and the starts begin (the MBRs: 0); all of it */
    explicit MeetLayout(size_t n) {
        cap = (n + MEET_ROUND - 1) / MEET_ROUND * MEET_ROUND;
        keys = cap * sizeof(uint4);
        starts = keys + cap * sizeof(unsigned long long);
        bytes = starts + cap * sizeof(uint32_t);
    }
};

/* a step's meetings in device memory, all to be read only */
struct Meets {
    const unsigned long long *keys;
    const uint32_t *starts;
    const uint4 *mbrs;
    __device__ inline unsigned long long key(uint64_t i) const { return keys[i]; }
    __device__ inline Bucket at(uint64_t i) const {
        const uint4 m = mbrs[i];
        return Bucket{keys[i], starts[i], {m.x, m.y, m.z, m.w}};
    }
};

/* a bucket that holds a live meeting (not a dead slot) */
__host__ __device__ inline bool bucket_live(const Bucket &b) { return (uint32_t)b.key != DEAD_B; }

__host__ __device__ inline uint32_t f2o(float f) {
    uint32_t b;
    memcpy(&b, &f, 4);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__host__ __device__ inline float o2f(uint32_t o) {
    uint32_t b = (o & 0x80000000u) ? (o & 0x7FFFFFFFu) : ~o;
    float f;
    memcpy(&f, &b, 4);
    return f;
}

/* float_to_uint (src/cuda/cuda_util.cuh:115-119): the quantised coordinate of
 * the per-object MBRs, saturating as the reference GPU converts */
__host__ __device__ inline uint32_t f2q(float xy) {
    xy += 180;
    float v = xy * 100000;
    if (!(v > 0.0f)) return 0;
    if (v >= 4294967296.0f) return 0xFFFFFFFFu;
    return (uint32_t)v;
}

#endif /* STC_TABLE_H_ */
