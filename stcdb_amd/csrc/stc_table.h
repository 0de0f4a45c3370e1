/*
 * stc_table.h — layout of the live meetings, shared by the pipeline and the
 * query kernels.
 *
 * A bucket is the reference's meeting_unit (src/tracing/workbench.h:62-83)
 * without its end time: 28 bytes of key, start and MBR. The MBR is stored as
 * order-preserving u32 images of the f32 bounds so that min/max updates are
 * integer ops. Keys are oid1 << 32 | oid2 with oid1 < oid2 < 2^26.
 *
 * The live meetings after a step are the buckets' keys, starts and MBRs, a
 * block of buckets after the other and in a block each of the three in a row
 * (a search by object then reads 8 bytes a meeting, not the lines of all 28: a
 * lookup among 10M meetings 52 -> 25 us), sorted by key, one
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

/* The meetings lie in blocks of MEET_BLOCK: a block's MBRs, its keys, its starts, each in a row, whole lines long. A
 * search by id reads the keys' rows alone (among 8.6M meetings as fast as from an array of keys), and the merge, which
 * reads and writes all, has one stream of memory on either side: a tile's new meetings are a block, 3.5 KB without a
 * gap. With the three as arrays of their own, gigabytes apart, the merge of 1.03e9 meetings took from 13.5 to 16.7 ms,
 * from process to process and from one of the two sets to the other; with 28-byte meetings one after the other 13.5
 * to 13.9; 13.5 to 14.3 so, and alike in both sets (blocks of 256 to 4,096: 13.7 to 14.7). */
#define MEET_BLOCK 128u
#define MEET_BLOCK_BYTES (MEET_BLOCK * 28u)
#define MEET_KEYS_AT (MEET_BLOCK * 16u)
#define MEET_STARTS_AT (MEET_BLOCK * 24u)

__host__ __device__ inline uint64_t meet_mbr_at(uint64_t i) { return i / MEET_BLOCK * MEET_BLOCK_BYTES + i % MEET_BLOCK * 16; }
__host__ __device__ inline uint64_t meet_key_at(uint64_t i) {
    return i / MEET_BLOCK * MEET_BLOCK_BYTES + MEET_KEYS_AT + i % MEET_BLOCK * 8;
}
__host__ __device__ inline uint64_t meet_start_at(uint64_t i) {
    return i / MEET_BLOCK * MEET_BLOCK_BYTES + MEET_STARTS_AT + i % MEET_BLOCK * 4;
}

/* a step's meetings in device memory, all to be read only */
struct Meets {
    const uint8_t *base;
    __device__ inline unsigned long long key(uint64_t i) const { return *(const unsigned long long *)(base + meet_key_at(i)); }
    __device__ inline uint32_t start(uint64_t i) const { return *(const uint32_t *)(base + meet_start_at(i)); }
    __device__ inline uint4 mbr(uint64_t i) const { return *(const uint4 *)(base + meet_mbr_at(i)); }
    __device__ inline Bucket at(uint64_t i) const {
        const uint4 m = mbr(i);
        return Bucket{key(i), start(i), {m.x, m.y, m.z, m.w}};
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
