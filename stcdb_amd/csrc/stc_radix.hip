/*
 * stc_radix.hip — stable LSD radix sort and prefix sums for gfx950.
 *
 * One pass per 8-bit digit:
 *   histogram : each workgroup counts the digits of its tile of keys in LDS;
 *   offsets   : a sort of up to 128 tiles lets every scatter workgroup add up
 *               the tiles' histograms itself; a larger one writes them
 *               digit-major (digit * tiles + tile) and scans each digit's row
 *               with a workgroup of its own, the 256 totals being added up by
 *               the scatter;
 *   scatter   : each workgroup ranks its tile stably and moves it. A wave holds
 *               its stretch of the tile in registers, all loads issued before
 *               the first ranking, and ranks it 64 keys a round by peer masks
 *               from 8 ballots and digit counts of its own in LDS, without a
 *               barrier; the waves' counts are added up once at the end. 4-byte
 *               keys are placed in LDS in digit order and written out in that
 *               order (coalesced), 8-byte keys straight to their global
 *               positions.
 * Keys of equal digit keep their input order, so chaining passes from the
 * least significant digit gives a stable sort, as thrust::sort_by_key on
 * primitive keys does in the reference (src/cuda/geometry.cu:1860, 1878-1886).
 *
 * What bounds it below a million keys is latency, so the tile is 1024 keys up
 * to 64k keys (a tile is then 4 rounds, and 50k keys are 49 workgroups instead
 * of 13), 2048 up to 2M and 4096 above. With 4096-key tiles ranked 256 keys a
 * round, four barriers and a load in each, a pass over 50k keys took five
 * launches and 27 us and takes two and 9 us so; one over 1M keys took six and
 * 37 us and takes three and 19 us (four and 22 with a scan of the whole table).
 */
#include "stc_internal.h"

#define RS_THREADS 256
#define RS_WAVES (RS_THREADS / STC_WAVE)
#define RS_BINS 256
#define RS_DIRECT 128          /* tiles whose histograms a scatter workgroup adds up itself */
#define RS_SMALL (64u << 10)   /* keys up to which a tile has 4 keys a thread */
#define RS_MEDIUM (2u << 20)   /* and 8 */
#define SCAN_THREADS 1024
#define SCAN_ITEMS 4
#define SCAN_TILE (SCAN_THREADS * SCAN_ITEMS)
#define SCAN_SUMS 4096         /* tile sums that a scan workgroup adds up itself */

static inline uint32_t ceil_div(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }
static inline uint32_t rs_items(uint32_t n) { return n <= RS_SMALL ? 4 : n <= RS_MEDIUM ? 8 : 16; }

size_t stc_radix_temp_words(uint32_t n) {
    if (!n) n = 1;
    /* histograms of a sort of up to n keys (the tiles of 2M keys outnumber those of a few more), then
     * the scans' tile sums, two levels */
    const uint32_t few = n < RS_MEDIUM ? n : RS_MEDIUM;
    const size_t t0 = ceil_div(n, RS_THREADS * 16), t1 = ceil_div(few, RS_THREADS * 8), t2 = RS_SMALL / (RS_THREADS * 4);
    const size_t hist = RS_BINS * (t0 > t1 ? (t0 > t2 ? t0 : t2) : (t1 > t2 ? t1 : t2));
    const size_t s1 = ceil_div(n > hist ? n : hist, SCAN_TILE);
    return hist + RS_BINS + s1 + ceil_div(s1, SCAN_TILE) + 64;
}

/* ---------------- exclusive scan ---------------- */

__device__ inline uint32_t wave_incl_scan(uint32_t v, int lane) {
#pragma unroll
    for (int o = 1; o < STC_WAVE; o <<= 1) {
        uint32_t u = __shfl_up(v, o, STC_WAVE);
        if (lane >= o) v += u;
    }
    return v;
}

/* block-wide exclusive scan of one value per thread; the block's total to every thread in *total */
__device__ inline uint32_t block_excl_scan(uint32_t v, uint32_t *total) {
    __shared__ uint32_t wsum[SCAN_THREADS / STC_WAVE], all;
    int lane = threadIdx.x & (STC_WAVE - 1), w = threadIdx.x / STC_WAVE;
    const int nw = (int)(blockDim.x / STC_WAVE);
    uint32_t inc = wave_incl_scan(v, lane);
    if (lane == STC_WAVE - 1) wsum[w] = inc;
    __syncthreads();
    if (w == 0) {
        uint32_t x = lane < nw ? wsum[lane] : 0;
        uint32_t xi = wave_incl_scan(x, lane);
        if (lane < nw) wsum[lane] = xi - x;
        if (lane == nw - 1) all = xi;
    }
    __syncthreads();
    uint32_t r = inc - v + wsum[w];
    *total = all;
    __syncthreads();
    return r;
}

__global__ __launch_bounds__(SCAN_THREADS) void k_scan_sums(const uint32_t *__restrict__ in, uint32_t n,
                                                             uint32_t *__restrict__ sums) {
    uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE + threadIdx.x;
    uint32_t s = 0, tot;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; k++) {
        const uint64_t i = base + (uint64_t)k * SCAN_THREADS;
        s += i < n ? in[i] : 0;
    }
    block_excl_scan(s, &tot);
    if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

/* One tile per workgroup: the tiles before it (their sums added up here, or
 * scanned already), then the tile. in may equal out. Up to SCAN_SUMS tiles the
 * scan is these two launches (before: one per level up and down, one for the
 * total and a copy of the last value; five for 1M values). */
__global__ __launch_bounds__(SCAN_THREADS) void k_scan_apply(const uint32_t *in, uint32_t *out, uint32_t n,
                                                              const uint32_t *__restrict__ sums, int scanned,
                                                              uint32_t *total) {
    const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE + (uint64_t)threadIdx.x * SCAN_ITEMS;
    uint32_t v[SCAN_ITEMS];
    uint32_t s = 0, before = 0, tot;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; k++) {
        v[k] = (base + k < n) ? in[base + k] : 0;
        s += v[k];
    }
    if (scanned) {
        before = sums[blockIdx.x];
    } else if (blockIdx.x) {
        uint32_t p = 0;
        for (uint32_t i = threadIdx.x; i < blockIdx.x; i += SCAN_THREADS) p += sums[i];
        block_excl_scan(p, &before);
    }
    uint32_t ex = before + block_excl_scan(s, &tot);
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; k++) {
        if (base + k < n) out[base + k] = ex;
        ex += v[k];
    }
    if (total && blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *total = before + tot;
}

static int scan_rec(const uint32_t *in, uint32_t *out, uint32_t n, uint32_t *total, uint32_t *temp, hipStream_t s) {
    const uint32_t tiles = ceil_div(n, SCAN_TILE);
    const bool two = tiles > SCAN_SUMS;
    if (tiles > 1) hipLaunchKernelGGL(k_scan_sums, dim3(tiles), dim3(SCAN_THREADS), 0, s, in, n, temp);
    if (two && scan_rec(temp, temp, tiles, nullptr, temp + tiles, s)) return -1;
    hipLaunchKernelGGL(k_scan_apply, dim3(tiles), dim3(SCAN_THREADS), 0, s, in, out, n, (const uint32_t *)temp, two ? 1 : 0, total);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int stc_exclusive_scan_u32(const uint32_t *in, uint32_t *out, uint32_t n, uint32_t *total_dev, uint32_t *temp,
                           hipStream_t s) {
    if (n == 0) {
        if (total_dev) hipMemsetAsync(total_dev, 0, 4, s);
        return 0;
    }
    if (scan_rec(in, out, n, total_dev, temp, s)) return stc_hip_fail(hipGetLastError(), "scan", __FILE__, __LINE__);
    return 0;
}

/* ---------------- radix passes ---------------- */

/* digit counts of each tile, tile after tile (by_tile) or digit-major */
template <typename K, int ITEMS>
__global__ __launch_bounds__(RS_THREADS) void k_rs_hist(const K *__restrict__ keys, uint32_t n, int shift,
                                                         uint32_t *__restrict__ hist, uint32_t tiles, int by_tile) {
    __shared__ uint32_t h[RS_BINS];
    h[threadIdx.x] = 0;
    const uint64_t base = (uint64_t)blockIdx.x * (RS_THREADS * ITEMS) + threadIdx.x;
    K k[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
        const uint64_t i = base + (uint64_t)r * RS_THREADS;
        k[r] = i < n ? keys[i] : (K)0;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; r++)
        if (base + (uint64_t)r * RS_THREADS < n) atomicAdd(&h[(uint32_t)(k[r] >> shift) & (RS_BINS - 1)], 1u);
    __syncthreads();
    hist[by_tile ? (uint64_t)blockIdx.x * RS_BINS + threadIdx.x : (uint64_t)threadIdx.x * tiles + blockIdx.x] = h[threadIdx.x];
}

/* Each digit's row of the digit-major table (a workgroup each) to the keys of
 * the digit in the tiles before, and the rows' totals. */
__global__ __launch_bounds__(RS_THREADS) void k_rs_rows(uint32_t *__restrict__ hist, uint32_t tiles, uint32_t *__restrict__ totals) {
    uint32_t *row = hist + (uint64_t)blockIdx.x * tiles;
    uint32_t before = 0;
    for (uint32_t t0 = 0; t0 < tiles; t0 += RS_THREADS * SCAN_ITEMS) {
        const uint32_t base = t0 + threadIdx.x * SCAN_ITEMS;
        uint32_t v[SCAN_ITEMS], s = 0, tot;
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; k++) {
            v[k] = base + k < tiles ? row[base + k] : 0;
            s += v[k];
        }
        uint32_t ex = before + block_excl_scan(s, &tot);
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; k++) {
            if (base + k < tiles) row[base + k] = ex;
            ex += v[k];
        }
        before += tot;
    }
    if (threadIdx.x == 0) totals[blockIdx.x] = before;
}

/* by_tile: offs holds the tiles' histograms; else the digit-major table of
 * k_rs_rows and behind it the totals. vin null: the values are the keys' places. */
template <typename K, int ITEMS>
__global__ __launch_bounds__(RS_THREADS) void k_rs_scatter(const K *__restrict__ kin, const uint32_t *__restrict__ vin,
                                                            K *__restrict__ kout, uint32_t *__restrict__ vout, uint32_t n,
                                                            int shift, const uint32_t *__restrict__ offs, uint32_t tiles,
                                                            int by_tile) {
    constexpr uint32_t TILE = RS_THREADS * ITEMS;
    constexpr bool STAGED = sizeof(K) == 4; /* an LDS tile of 8-byte keys would cost the kernel its occupancy */
    __shared__ uint32_t base[RS_BINS];   /* global position of the tile's first key of each digit, less its place in LDS */
    __shared__ uint32_t wcnt[RS_WAVES][RS_BINS];
    __shared__ K sk[STAGED ? TILE : 1];
    __shared__ uint32_t sv[STAGED ? TILE : 1];
    const int tid = threadIdx.x, lane = tid & (STC_WAVE - 1), w = tid / STC_WAVE;
    const uint64_t tile0 = (uint64_t)blockIdx.x * TILE;
    const uint64_t first = tile0 + (uint64_t)w * (STC_WAVE * ITEMS) + lane; /* the wave's stretch, 64 keys a round */
    K k[ITEMS];
    uint32_t v[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
        const uint64_t i = first + (uint64_t)r * STC_WAVE;
        k[r] = i < n ? kin[i] : (K)0;
        v[r] = vin ? (i < n ? vin[i] : 0u) : (uint32_t)i;
    }
#pragma unroll
    for (int q = 0; q < RS_WAVES; q++) wcnt[q][tid] = 0;
    /* where the tile's keys of digit tid start */
    uint32_t b0, tot;
    if (by_tile) {
        uint32_t pre = 0, all = 0;
#pragma unroll 16
        for (uint32_t t = 0; t < tiles; t++) {
            const uint32_t c = offs[t * RS_BINS + tid];
            all += c;
            pre += t < blockIdx.x ? c : 0u;
        }
        b0 = pre + block_excl_scan(all, &tot);
    } else {
        const uint32_t pre = offs[(uint64_t)tid * tiles + blockIdx.x];
        b0 = pre + block_excl_scan(offs[(uint64_t)RS_BINS * tiles + tid], &tot);
    }
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (STC_WAVE - lane));
    uint32_t rank[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
        const bool valid = first + (uint64_t)r * STC_WAVE < n;
        const uint32_t d = (uint32_t)(k[r] >> shift) & (RS_BINS - 1);
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const bool bit = (d >> b) & 1u;
            const uint64_t m = __ballot(bit);
            peers &= bit ? m : ~m;
        }
        const uint32_t behind = (uint32_t)__popcll(peers & lt);
        const uint32_t seen = wcnt[w][d];
        rank[r] = seen + behind;
        /* the wave's own counts: its lanes' reads come before the write, its LDS accesses in order */
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (valid && behind == 0) wcnt[w][d] = seen + (uint32_t)__popcll(peers);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    uint32_t acc = 0;
#pragma unroll
    for (int q = 0; q < RS_WAVES; q++) {
        const uint32_t c = wcnt[q][tid];
        wcnt[q][tid] = acc;
        acc += c;
    }
    if constexpr (STAGED) {
        const uint32_t l0 = block_excl_scan(acc, &tot);
        base[tid] = b0 - l0;
#pragma unroll
        for (int q = 0; q < RS_WAVES; q++) wcnt[q][tid] += l0;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < ITEMS; r++)
            if (first + (uint64_t)r * STC_WAVE < n) {
                const uint32_t at = wcnt[w][(uint32_t)(k[r] >> shift) & (RS_BINS - 1)] + rank[r];
                sk[at] = k[r];
                sv[at] = v[r];
            }
        __syncthreads();
        const uint32_t cnt = (uint32_t)min<uint64_t>(TILE, n - tile0);
        for (uint32_t p = tid; p < cnt; p += RS_THREADS) {
            const K key = sk[p];
            const uint32_t pos = base[(uint32_t)(key >> shift) & (RS_BINS - 1)] + p;
            kout[pos] = key;
            vout[pos] = sv[p];
        }
    } else {
        base[tid] = b0;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < ITEMS; r++)
            if (first + (uint64_t)r * STC_WAVE < n) {
                const uint32_t d = (uint32_t)(k[r] >> shift) & (RS_BINS - 1);
                const uint32_t pos = base[d] + wcnt[w][d] + rank[r];
                kout[pos] = k[r];
                vout[pos] = v[r];
            }
    }
}

template <typename K, int ITEMS>
static int radix_pass(const K *kin, const uint32_t *vin, K *kout, uint32_t *vout, uint32_t n, int shift, uint32_t *temp,
                      hipStream_t s) {
    const uint32_t tiles = ceil_div(n, RS_THREADS * ITEMS);
    const int by_tile = tiles <= RS_DIRECT;
    hipLaunchKernelGGL((k_rs_hist<K, ITEMS>), dim3(tiles), dim3(RS_THREADS), 0, s, kin, n, shift, temp, tiles, by_tile);
    STC_CHECK(hipGetLastError());
    if (!by_tile) {
        hipLaunchKernelGGL(k_rs_rows, dim3(RS_BINS), dim3(RS_THREADS), 0, s, temp, tiles, temp + (size_t)RS_BINS * tiles);
        STC_CHECK(hipGetLastError());
    }
    hipLaunchKernelGGL((k_rs_scatter<K, ITEMS>), dim3(tiles), dim3(RS_THREADS), 0, s, kin, vin, kout, vout, n, shift,
                       (const uint32_t *)temp, tiles, by_tile);
    STC_CHECK(hipGetLastError());
    return 0;
}

template <typename K>
static int radix_sort(const K *kin, const uint32_t *vin, K *keys, uint32_t *vals, K *keys_alt, uint32_t *vals_alt,
                      uint32_t n, int lo_bit, int hi_bit, uint32_t *temp, bool *in_alt, hipStream_t s) {
    *in_alt = false;
    const bool in_place = kin == keys;
    if (n == 0 || (in_place && vin && (n == 1 || hi_bit <= lo_bit))) return 0;
    const K *src_k = kin;
    const uint32_t *src_v = vin;
    bool to_alt = in_place;
    for (int shift = lo_bit; shift < hi_bit || shift == lo_bit; shift += 8, to_alt = !to_alt) {
        K *dk = to_alt ? keys_alt : keys;
        uint32_t *dv = to_alt ? vals_alt : vals;
        const uint32_t items = rs_items(n);
        const int rc = items == 4   ? radix_pass<K, 4>(src_k, src_v, dk, dv, n, shift, temp, s)
                       : items == 8 ? radix_pass<K, 8>(src_k, src_v, dk, dv, n, shift, temp, s)
                                    : radix_pass<K, 16>(src_k, src_v, dk, dv, n, shift, temp, s);
        if (rc) return rc;
        src_k = dk;
        src_v = dv;
        *in_alt = to_alt;
    }
    return 0;
}

int stc_radix_sort_u32(const uint32_t *kin, const uint32_t *vin, uint32_t *keys, uint32_t *vals, uint32_t *keys_alt,
                       uint32_t *vals_alt, uint32_t n, int bits, uint32_t *temp, bool *in_alt, hipStream_t s) {
    return radix_sort<uint32_t>(kin, vin, keys, vals, keys_alt, vals_alt, n, 0, bits, temp, in_alt, s);
}

int stc_radix_sort_u64(const uint64_t *kin, const uint32_t *vin, uint64_t *keys, uint32_t *vals, uint64_t *keys_alt,
                       uint32_t *vals_alt, uint32_t n, int lo_bit, int hi_bit, uint32_t *temp, bool *in_alt, hipStream_t s) {
    return radix_sort<uint64_t>(kin, vin, keys, vals, keys_alt, vals_alt, n, lo_bit, hi_bit, temp, in_alt, s);
}
