// yoco_z1: the owner's token-embedding gradient (declarations: include/yoco_z1.h).
//
// Replaces torch.ops.aten.embedding_dense_backward(g_all, ids, V, padding_idx, False) on the embedding's owner,
// followed or preceded by the x 1/world of the reference (yoco/models/decoder/layer_graphs.py:87-93,
// yoco/models/decoder/ce_reduce.py:226-231).  Same summation order as aten for the row count.  For more than 3072
// indices aten sorts: occurrences of each token id in stable position order, fp32 partial sums over runs of 10
// consecutive occurrences, the partials summed in order, one rounding to bf16.  For fewer its other kernel walks
// the indices in chunks of 16: per chunk and id an fp32 sum in position order, rounded to bf16 and added to the
// bf16 row.  padding_idx rows and ids outside [0, V) contribute nothing.
//
//   1. each id's occurrences in position order -- ent, all of an id's next to each other -- and info[t], where those of
//      id t are and how many: for up to kBucketRows rows one launch, emb_bucket_kernel; beyond, keys[i] = id_i (or V when
//      out of range) and vals[i] = i sorted stably by key -- hipCUB's radix sort, or, while the stream is being captured
//      into a HIP graph, rocPRIM's merge sort, which clears nothing with memsets (the radix sort does; both are stable,
//      so the order is the same) -- and binary searches over the sorted keys, one per t and one per place;
//   2. emb_rows_kernel writes every row of the table exactly once (aten zero-fills the whole table and then scatters
//      into it): first waves for the runs of ids with many occurrences, then one wave per row, in order, which zeroes
//      it or sums its few occurrences.  Token frequencies in text are skewed: one wave (or one workgroup) walking
//      thousands of occurrences of one id would take milliseconds;
//   3. emb_chain_kernel adds the run partials of each id with several, in run order per column.
// (For few indices a run is an id's occurrences in one chunk of 16 indices.)
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>
#include <rocprim/device/device_merge_sort.hpp>

#include <stdint.h>

#include <type_traits>

#include "yoco_z1.h"
#include "z1_internal.h"

#pragma clang fp contract(off)

namespace {

constexpr int kEmbThreads = 64;                  // one wave per output row
constexpr int kRowsPerPartial = 10;        // aten's NROWS_PER_THREAD
// aten sorts for more than kSortMinRows - 1 indices; for fewer its kernel walks the indices in chunks of
// kFewRowsChunk (torch's ROCm build; checked bit for bit against it on MI355X)
constexpr int64_t kSortMinRows = 3073;
constexpr int kFewRowsChunk = 16;
constexpr int kWave = 64;
// The rows launch.  Figures: whole calls on 16,384 rows of 3072 into a 100,288-row table, gradients not cached, uniform /
// Zipf(1.2) ids; 141 / 153 us as it stands, 141 / 152 when they were taken.
// Resident workgroups per CU, capped with a dynamic LDS reservation the kernel does not use: 141 / 153 at 14, 143 / 152 at
// 20, 152 / 157 at 10, 175 / 185 at 8 (a short table, 2000 rows of 768 into 32,000: 32.4 us at 20, 33.9 at 14, 37 at 10).
// Dense tables (below) run as many as fit: they read more than they write, in waves that sum up to 20 rows.  At 16 / all:
// 100,000 of 768 into 32,000 rows 117.9 / 108.0 and 157.8 / 148.6, 50,000 of 768 into 256 88.7 / 81.5 and 104.5 / 98.4, 1.2M
// of 768 into 32,000 879 / 813 and 1033 / 976, 50,000 of 64 into 8000 61.0 / 59.4 and 88.4 / 90.0.
constexpr int kEmbWgPerCu = 16;
constexpr int kDirect = 4;                 // most occurrences of an id that the wave of its row sums (2: the same)
// In a dense table, of kDenseMean indices per row or more on average, the wave of a row sums up to kDirectDense occurrences
// (two runs): most ids have between 5 and 20 there, and the row waves alone fill the chip, so that partials sent through
// memory only add traffic.  Whole calls, gradients not cached, run by run / by the row's wave (us, uniform and Zipf(1.2)
// ids, both at kEmbWgPerCu): 1.2M indices of width 768 into 100,288 rows 1376 / 557 and 1160 / 1139; 256,000 of 768 into
// 32,000 rows 305 / 204 and 340 / 332; 64,000 of 3072 into 32,000 rows 209 / 183 and 227 / 214; 32,000 of 768 into 8000 rows
// 42 / 38 and 70 / 69. With 1.5 indices per row 48,000 of 768 take 56 / 57 us.  Fewer indices than kDenseRows leave long
// waves alone on the chip: 12,000 Zipf ones of 3072 into 1000 rows 49 / 53 us, 20,000 80 / 77 us.
constexpr int kDirectDense = 2 * kRowsPerPartial;
constexpr int64_t kDenseMean = 2;
constexpr int64_t kDenseRows = 16384;
constexpr int kRunBlock = 40;              // sorted positions whose runs a wave sums, for one step of 512 columns
// In a dense table of this many indices per row or more most ids are summed by runs, and shorter blocks give more waves:
// half the length (at kEmbWgPerCu: 65,536 ids of width 256 into 256 rows, uniform / Zipf, 78.5 / 107.4 us with 40, 72.1 /
// 101.8 with 20; 131,072 of 768 into 1000 rows 152 / 195 and 147 / 187; at 8 per row it loses: 262,144 of 768 into 32,000
// rows 205 / 334 and 209 / 337), and a quarter where a half gives at most kQuarterWaves waves: 20,000 of 256 into 256 rows
// 37.4 / 48.6 and 34.3 / 45.6, 100,000 of 64 (5000 waves) 85.8 / 122.1 and 83.8 / 119.6, but 20,000 of 3072 (6000) 64.6 /
// 75.7 and 66.9 / 83.2.
constexpr int64_t kShortBlockMean = 16;
constexpr int64_t kQuarterWaves = 5120;
constexpr int kFewBlock = 8;               // the same, few indices
constexpr int kMaxWaves = 1 << 20;         // most waves that sum runs (they stride beyond that)
// Consecutive rows of one XCD: spans of 32 to 128 rows measure alike, single rows round robin 144 / 153; one eighth of the
// table each leaves the frequent ids, which are the first ones, to one XCD.
constexpr int kSpan = 128;
constexpr int64_t kMaxRowWaves = 1 << 25;   // a multiple of 8 kSpan; with kMaxWaves within one launch's 2^32 threads
// Cache-policy bits of the rows' stores, sc0 sc1 nt as the update's streams have: 141 / 154 us against 147 / 158 with nt
// alone, 159 / 164 with sc0 sc1, 161 / 164 with none.  (Waves that only zero and waves that only sum, in one launch in
// either order or mixed, 141-161 / 160-173: a row-ordered mix suits the DRAM better than two patterns at once.)
constexpr int kRowPolicy = 1 | 2 | 16;
// An id with more than kDirect occurrences is summed run by run.  If it has several runs, their partials go to slots:
// run k of an id whose occurrences start at sorted position lo to slot ceil(lo / kSlotSpan) + k.  Its n >= 11
// occurrences have ceil(n / 10) runs and at least (n - 6) / 4 whole slots of their own, which is never fewer.  (At most
// kSortMinRows - 1 rows, where a run may be a single occurrence: slot = its sorted position.)
constexpr int kSlotSpan = 4;
static_assert(kRowsPerPartial == 10 && kSlotSpan == 4 && kDirect <= kRowsPerPartial, "slots of different ids are disjoint");
constexpr int kChainWaves = 16;            // chain pass: waves that load a batch of partials
constexpr int kChainDepth = 16;            // partials per lane per batch (64 KB of LDS)
constexpr int kChainRows = kChainWaves * kChainDepth;
static_assert(kChainRows % 16 == 0, "wave 0 reads a batch 16 rows at a time");
constexpr int kFewRuns = (int)(kSortMinRows + kFewRowsChunk - 2) / kFewRowsChunk;    // most runs of an id, few indices
static_assert(kFewRuns % kChainWaves == 0, "each wave loads as many");
constexpr int kChainGrid = 512;
constexpr int kWaveChainRuns = 32;         // ids of at most this many runs are chained by one wave
constexpr int64_t kMaxCols = 1 << 24;      // D limit: keeps the workspace size and offsets far from overflow

__device__ __forceinline__ float bf16f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// Round to nearest even, with gfx950's conversion (a NaN keeps its sign and payload: finish makes aten's of it).
__device__ __forceinline__ uint16_t bf16r(float x) { return __builtin_bit_cast(uint16_t, (__bf16)x); }

// One place of the order (each id's occurrences next to each other, by position): the occurrence's position, its id, and
// the id's first place and count.
struct Ent {
    int32_t pos;
    uint32_t id;
    int32_t lo, n;
};
static_assert(sizeof(Ent) == 16, "one 16-byte load");

__global__ void emb_keys_kernel(const int64_t* __restrict__ ids, int64_t R, int64_t V, uint32_t* __restrict__ keys,
                                int32_t* __restrict__ vals) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= R) return;
    const int64_t t = ids[i];
    keys[i] = (t >= 0 && t < V) ? (uint32_t)t : (uint32_t)V;
    vals[i] = (int32_t)i;
}

// info[t] = (where, count) of id t's occurrences, for t in [0, V): their first sorted place, or the position of the
// only one.  Independent binary searches over the sorted keys, one thread per t (the latency of the searches overlaps),
// for both ends of t's occurrences side by side (one after the other 7.6 us for 65,536 keys, 5.4 for one end alone).
__device__ __forceinline__ int2 key_range(const uint32_t* __restrict__ sorted, int64_t R, uint32_t key) {
    int lo = 0, hi = 0;                         // the first places of keys >= key and > key lie in [lo, lo + n], [hi, hi + n]
    for (int n = (int)R; n > 0;) {
        const int half = n >> 1;
        const uint32_t a = sorted[lo + half], b = sorted[hi + half];
        if (a < key) lo += n - half;
        if (b <= key) hi += n - half;
        n = half;
    }
    return int2{lo, hi};
}

// info, and ent of every sorted place: the first `vocab_blocks` workgroups have a thread per id, the others (up to
// kSearchRows indices) one per place, which searches for its own id's range rather than wait for info in a launch of its
// own.  Whole calls, two launches / one: 50,000 indices of width 64 into 8000 rows 63.1 / 61.1 us, 100,000 87.0 / 85.0,
// 200,000 of 768 into 32,000 rows 149.9 / 149.3; 262,144 are even, and 500,000 of 256 take 256.6 / 262.5, 1.2M of 64 into
// 8000 rows 318 / 326: a search per place then costs more than a launch.
constexpr int64_t kSearchRows = 1 << 18;
constexpr int kPlaceThreads = 256;
__global__ __launch_bounds__(kPlaceThreads) void emb_places_kernel(const uint32_t* __restrict__ sorted,
                                                                   const int32_t* __restrict__ spos, int64_t R, int64_t V,
                                                                   int vocab_blocks, int2* __restrict__ info,
                                                                   Ent* __restrict__ ent, int* __restrict__ counts) {
    if (blockIdx.x == 0 && threadIdx.x < 2) counts[threadIdx.x] = 0;   // the rows kernel appends to the lists after this
    if ((int)blockIdx.x < vocab_blocks) {
        const int64_t t = (int64_t)blockIdx.x * kPlaceThreads + threadIdx.x;
        if (t >= V) return;
        const int2 r = key_range(sorted, R, (uint32_t)t);
        info[t] = int2{r.y - r.x == 1 ? spos[r.x] : r.x, r.y - r.x};
        if (t == V - 1) counts[2] = r.y;        // the ids inside [0, V)
        return;
    }
    const int64_t p = (int64_t)((int)blockIdx.x - vocab_blocks) * kPlaceThreads + threadIdx.x;
    if (p >= R) return;
    const uint32_t id = sorted[p];
    if ((int64_t)id >= V) return;
    const int2 r = key_range(sorted, R, id);
    ent[p] = Ent{spos[p], id, r.x, r.y - r.x};
}

// ent of every sorted place, from info.
__global__ __launch_bounds__(kPlaceThreads) void emb_entries_kernel(const uint32_t* __restrict__ sorted,
                                                                    const int32_t* __restrict__ spos, int64_t R, int64_t V,
                                                                    const int2* __restrict__ info, Ent* __restrict__ ent) {
    const int64_t p = (int64_t)blockIdx.x * kPlaceThreads + threadIdx.x;
    if (p >= R) return;
    const uint32_t id = sorted[p];
    if ((int64_t)id >= V) return;
    const int2 r = info[id];
    ent[p] = Ent{spos[p], id, r.y == 1 ? (int32_t)p : r.x, r.y};
}

// The same results (ent and info) in one launch, without a sort over the whole list.  The ids are
// split over 2^kb buckets, granules of 2^kGranuleBits consecutive ids round robin, one workgroup per bucket (text's
// frequent ids are the small ones: spread, no workgroup gets them all); round h begins at bucket turn * h, so that ids a
// multiple of the round apart do not meet in one bucket either.  Every workgroup reads all R ids, wave w the
// w-th segment: it counts its bucket's ids per wave and local id in LDS (l: the id's number within the bucket) and how
// many ids belong to smaller buckets, which is where its range of the sorted order starts; prefix sums over the waves
// of one id, then over the ids, give every (wave, id) its place; then each wave places its occurrences in position
// order, lanes with the same id by rank.  No workgroup waits for another, no atomic decides an order, nothing has to be
// cleared beforehand.  Latency bounds it: two rounds over the wave's ids (kept in registers when they are one tile) and
// three barriers, and for a frequent id the rounds of its bucket's placement.
// Measured in whole calls of width 64 into 100,288 rows (uniform / Zipf(1.2) ids), against the five to seven launches
// of keys, library sort and searches: 500 rows 37 / 45 against 43 / 51 us, 4096 42 / 52 against 55 / 66, 16,384
// 48 / 70 against 71 / 89, 65,536 98 / 143 against 104 / 144, 131,072 148 / 231 against 136 / 203; the reading of all
// ids by every workgroup grows with R, hence kBucketRows.  Granules of 8 ids put 8 frequent ids into one bucket (Zipf
// 80 us at 16,384 rows), single ids scatter info in 8-byte writes (52 / 71 us); fewer than 2^8 buckets leave
// small vocabularies to a few workgroups (2000 rows: 57 us with 8, 41 us with 256).
constexpr int kBucketThreads = 1024;
constexpr int kBucketWaves = kBucketThreads / kWave;
constexpr int kBucketTile = 16;            // ids per lane and tile
constexpr int kGranuleBits = 1;
constexpr int kMaxLocal = 512;             // local ids of a bucket: kBucketWaves x 512 counters, 32 KB of LDS
constexpr int kMinBucketBits = 8;
constexpr int kMaxBucketBits = 10;
constexpr int64_t kBucketRows = 49152;
constexpr int64_t kBucketVocab = (int64_t)kMaxLocal << kMaxBucketBits;
// The turn: 2^kb over the golden ratio, made odd.  16,384 / 49,152 ids into 100,288 rows of 768, whole calls: multiples of 512
// 52 / 90 us against 159 / 411 without turns, Zipf ids 60 / 111 against 59 / 111, uniform ones 49.4 / 82.4 against 49.2 / 80.0.
__device__ __forceinline__ uint32_t bucket_turn(int kb) { return (40503u >> (16 - kb)) | 1u; }

__global__ __launch_bounds__(kBucketThreads) void emb_bucket_kernel(const int64_t* __restrict__ ids, int R, int V,
                                                                    int kb, Ent* __restrict__ ent,
                                                                    int2* __restrict__ info,
                                                                    int* __restrict__ counts) {
    __shared__ int hist[kBucketWaves][kMaxLocal];
    __shared__ int2 range[kMaxLocal];        // a local id's first place and count
    __shared__ int wsum[kBucketWaves], wless[kBucketWaves];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
    const int k = blockIdx.x, mask = (1 << kb) - 1;
    const uint32_t turn = bucket_turn(kb);
    if (k == 0 && threadIdx.x < 2) counts[threadIdx.x] = 0;   // the rows kernel appends to the lists after this
    for (int i = lane; i < kMaxLocal; i += kWave) hist[wave][i] = 0;        // this wave's own counters
    // a wave's segment: positions [s0, s1), 64 consecutive ones a step
    const int steps = (R + kBucketThreads - 1) / kBucketThreads;
    const int s0 = wave * steps * kWave, s1 = s0 + steps * kWave < R ? s0 + steps * kWave : R;
    int loc[kBucketTile];                    // local id, -1: another bucket's (or out of range)
    int less = 0;
    auto id_of = [&](int l) {                // the id with local id l
        const int h = l >> kGranuleBits;
        return (((h << kb) | ((k - (int)turn * h) & mask)) << kGranuleBits) | (l & ((1 << kGranuleBits) - 1));
    };
    auto load = [&](int p0) {                // the tile at p0; returns how many of the lane's ids are in smaller buckets
        int64_t t[kBucketTile];
#pragma unroll
        for (int i = 0; i < kBucketTile; ++i) {
            const int p = p0 + i * kWave + lane;
            t[i] = p < s1 ? ids[p] : -1;
        }
        int c = 0;
#pragma unroll
        for (int i = 0; i < kBucketTile; ++i) {
            const bool ok = (uint64_t)t[i] < (uint64_t)V;
            const uint32_t id = (uint32_t)t[i], h = id >> (kGranuleBits + kb);
            const int b = (int)((__umul24(h, turn << kGranuleBits) + id) >> kGranuleBits) & mask;
            loc[i] = ok && b == k ? (int)((h << kGranuleBits) | (id & ((1 << kGranuleBits) - 1))) : -1;
            c += ok && b < k;
        }
        return c;
    };
    for (int p0 = s0; p0 < s1; p0 += kBucketTile * kWave) {
        less += load(p0);
#pragma unroll
        for (int i = 0; i < kBucketTile; ++i)
            if (loc[i] >= 0) atomicAdd(&hist[wave][loc[i]], 1);
    }
    for (int off = kWave / 2; off > 0; off >>= 1) less += __shfl_xor(less, off);
    if (lane == 0) wless[wave] = less;
    __syncthreads();
    // thread l: local id l's occurrences wave by wave, then its start among the bucket's ids
    const int l = threadIdx.x;
    int cnt = 0;
    if (l < kMaxLocal) {
        int c[kBucketWaves];
#pragma unroll
        for (int w = 0; w < kBucketWaves; ++w) c[w] = hist[w][l];
#pragma unroll
        for (int w = 0; w < kBucketWaves; ++w) {
            hist[w][l] = cnt;
            cnt += c[w];
        }
    }
    int incl = cnt;
    for (int off = 1; off < kWave; off <<= 1) {
        const int x = __shfl_up(incl, off);
        if (lane >= off) incl += x;
    }
    if (lane == kWave - 1) wsum[wave] = incl;
    __syncthreads();
    int start = incl - cnt;
    for (int w = 0; w < kBucketWaves; ++w) start += wless[w] + (w < wave ? wsum[w] : 0);
    if (k == mask && threadIdx.x == kBucketThreads - 1) counts[2] = start + cnt;    // the ids inside [0, V)
    if (l < kMaxLocal) {
#pragma unroll
        for (int w = 0; w < kBucketWaves; ++w) hist[w][l] += start;
        const int t = id_of(l);
        range[l] = int2{start, cnt};
        if (t < V && cnt != 1) info[t] = int2{start, cnt};
    }
    __syncthreads();
    const bool one_tile = steps <= kBucketTile;
    for (int p0 = s0; p0 < s1; p0 += kBucketTile * kWave) {
        if (!one_tile) load(p0);
#pragma unroll
        for (int i = 0; i < kBucketTile; ++i) {
            uint64_t left = __ballot(loc[i] >= 0);
            while (left) {                   // one id of the wave's 64 positions at a time, its lanes in order
                const int leader = __builtin_ctzll(left);
                const int l0 = __builtin_amdgcn_readlane(loc[i], leader);
                const bool mine = loc[i] == l0;
                const uint64_t same = __ballot(mine);
                const int at = hist[wave][l0];
                const int2 r = range[l0];
                const int id = id_of(l0);
                if (mine) {
                    const int p = p0 + i * kWave + lane;
                    ent[at + __builtin_popcountll(same & ((1ull << lane) - 1))] = Ent{p, (uint32_t)id, r.x, r.y};
                    if (r.y == 1) info[id] = int2{p, 1};
                }
                hist[wave][l0] = at + __builtin_popcountll(same);          // every lane, the same value
                left &= ~same;
            }
        }
    }
}

typedef uint32_t u4 __attribute__((ext_vector_type(4)));

// One gradient element as it enters a partial: scale_mode 1 rounds bf16(g * scale) first (the CE path scales the
// staged rows in place, ce_reduce.py:228).
__device__ __forceinline__ float grad_elem(uint16_t h, float scale, int scale_mode) {
    float v = bf16f(h);
    if (scale_mode == 1) v = bf16f(bf16r(v * scale));
    return v;
}

// The finished fp32 sum to bf16; scale_mode 2 multiplies the bf16 result by scale and rounds again
// (layer_graphs.py:93).  Every NaN comes out as 0x7fc0, the one aten's conversion gives.
__device__ __forceinline__ float scaled(float acc, float scale, int scale_mode) {
    return scale_mode == 2 ? bf16f(bf16r(acc)) * scale : acc;
}

__device__ __forceinline__ uint16_t finish(float acc, float scale, int scale_mode) {
    const float v = scaled(acc, scale, scale_mode);
    return v != v ? (uint16_t)0x7fc0u : bf16r(v);
}

// Rows start wherever t * D puts them: the wide accesses below assume 2-byte alignment only (gfx950 loads and stores 16
// bytes at any address; an odd D costs the lines that straddle).
typedef u4 u4_any __attribute__((aligned(2)));

__device__ __forceinline__ u4 load8(const uint16_t* p) {
    return *(const __attribute__((address_space(1))) u4_any*)p;
}
__device__ __forceinline__ void nt_store8(uint16_t* p, u4 x) {
    __builtin_nontemporal_store((u4_any)x, (__attribute__((address_space(1))) u4_any*)p);
}

// Stores to one row of the table: 16 bytes at byte offset off of orow (the same in the whole wave).  Rows on 16-byte
// boundaries (wide) take buffer stores marked kRowPolicy; others plain nontemporal ones.
__device__ __forceinline__ void row_store8(uint16_t* orow, bool wide, int bytes, int off, u4 x) {
    if (wide)
        __builtin_amdgcn_raw_buffer_store_b128(x, __builtin_amdgcn_make_buffer_rsrc(orow, 0, bytes, 0x00020000), off, 0,
                                               kRowPolicy);
    else
        nt_store8(orow + off / 2, x);
}

// Adds a finished partial to the row's sum: aten's sort path adds fp32 partials; its few-indices kernel rounds the
// partial to bf16 and the row after the add.
template <bool FEW>
__device__ __forceinline__ float add_part(float acc, float part) {
    return FEW ? bf16f(bf16r(acc + bf16f(bf16r(part)))) : acc + part;
}

// Whether the occurrence at sorted place p (position pos) of an id starting at lo begins a run: every 10th one, or, for
// few indices, the first one in its chunk of 16 positions (prev: the position at place p - 1, read where p > lo).
template <bool FEW>
__device__ __forceinline__ bool run_starts(int p, int lo, int pos, int prev) {
    return p == lo || (FEW ? pos / kFewRowsChunk != prev / kFewRowsChunk : (p - lo) % kRowsPerPartial == 0);
}

template <bool FEW>
__device__ __forceinline__ int64_t run_slot(int lo, int p) {
    return FEW ? p : ((int64_t)lo + kSlotSpan - 1) / kSlotSpan + (p - lo) / kRowsPerPartial;
}

// Eight finished sums.  One compare looks for a NaN in two of them, and lanes without one skip the rest.
__device__ __forceinline__ u4 finish8(const float (&acc)[8], float scale, int scale_mode) {
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = scaled(acc[k], scale, scale_mode);
    bool nan = false;
#pragma unroll
    for (int k = 0; k < 8; k += 2) nan |= __builtin_isunordered(v[k], v[k + 1]);
    if (nan) {
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = v[k] != v[k] ? __uint_as_float(0x7fc00000u) : v[k];
    }
    u4 o;
#pragma unroll
    for (int k = 0; k < 8; k += 2) o[k >> 1] = (uint32_t)bf16r(v[k]) | ((uint32_t)bf16r(v[k + 1]) << 16);
    return o;
}

__device__ __forceinline__ uint16_t col(const u4& x, int k) { return (uint16_t)(x[k >> 1] >> ((k & 1) * 16)); }

typedef float f4 __attribute__((ext_vector_type(4)));
typedef f4 f4_any __attribute__((aligned(4)));

// The runs that start at sorted places [p0, p0 + block) and belong to ids of more than DIRECT occurrences, columns
// [512 step, 512 (step + 1)) of each; the wave of the last step also takes the last D % 8 columns, one per lane.  A
// run's rows (at most 10, or 16 for few indices) are loaded together and summed in order.  The sum of an id's only run
// is its row; otherwise the fp32 partial goes to the run's slot, and the wave of step 0 lists the id for the chain pass.
template <bool FEW, int DIRECT>
__device__ __forceinline__ void sum_runs(int64_t p0, int block, int step, bool last_step,
                                         const uint16_t* __restrict__ grad, int64_t D, const Ent* __restrict__ ent,
                                         int64_t padding_idx, float scale, int scale_mode, int64_t valid,
                                         uint16_t* __restrict__ out, int* __restrict__ counts,
                                         int32_t* __restrict__ short_list, int32_t* __restrict__ long_list,
                                         float* __restrict__ parts) {
    constexpr int kRows = FEW ? kFewRowsChunk : kRowsPerPartial;
    static_assert(1 + (FEW ? kFewBlock : kRunBlock) + kRows <= kWave, "lanes for every place a run of the block reaches");
    const int lane = threadIdx.x;
    // lane i: place p0 - 1 + i
    const int64_t p = p0 - 1 + lane;
    Ent e = Ent{0, 0, 0, 0};
    if (p >= 0 && p < valid && lane < 1 + block + kRows) e = ent[p];
    const int prev = __shfl_up(e.pos, 1);
    const bool begins = p >= e.lo && e.n > 0 && run_starts<FEW>((int)p, e.lo, e.pos, prev);
    const bool mine = begins && lane >= 1 && lane <= block && e.n > DIRECT && (int64_t)e.id != padding_idx;
    const bool single = !FEW && e.n <= kRowsPerPartial;
    if (mine && !single && p == e.lo && step == 0) {
        const bool is_short = (FEW ? e.n : (e.n + kRowsPerPartial - 1) / kRowsPerPartial) <= kWaveChainRuns;
        (is_short ? short_list : long_list)[atomicAdd(&counts[is_short ? 0 : 1], 1)] = e.lo;
    }
    const int64_t ng = D / 8, gi = (int64_t)step * kEmbThreads + lane;
    for (uint64_t left = __ballot(mine), starts = __ballot(begins); left; left &= left - 1) {
        const int l = __builtin_ctzll(left);
        const int lo = __builtin_amdgcn_readlane(e.lo, l), n = __builtin_amdgcn_readlane(e.n, l), s = (int)p0 - 1 + l;
        // its rows: up to the next run's start or the id's end
        const uint64_t next = starts >> 1 >> l;
        int cnt = next ? 1 + __builtin_ctzll(next) : kRows;
        if (lo + n - s < cnt) cnt = lo + n - s;
        if (cnt > kRows) cnt = kRows;
        const int64_t row = (int64_t)__builtin_amdgcn_readlane((int)e.id, l) & 0xffffffff;
        const bool only = !FEW && n <= kRowsPerPartial;
        float* dst = parts + (only ? 0 : run_slot<FEW>(lo, s)) * D;
        int at[kRows];               // read with every lane active: lanes without a group hold places too
#pragma unroll
        for (int u = 0; u < kRows; ++u) at[u] = __builtin_amdgcn_readlane(e.pos, l + u);
        if (gi < ng) {
            u4 x[kRows];
#pragma unroll
            for (int u = 0; u < kRows; ++u)
                if (u < cnt) x[u] = load8(grad + (int64_t)at[u] * D + gi * 8);
            float part[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) part[k] = 0.0f;
#pragma unroll
            for (int u = 0; u < kRows; ++u) {
                if (u < cnt) {
#pragma unroll
                    for (int k = 0; k < 8; ++k) part[k] = part[k] + grad_elem(col(x[u], k), scale, scale_mode);
                }
            }
            if (only) {
#pragma unroll
                for (int k = 0; k < 8; ++k) part[k] = 0.0f + part[k];
                nt_store8(out + row * D + gi * 8, finish8(part, scale, scale_mode));
            } else {
                f4_any* o = reinterpret_cast<f4_any*>(dst + gi * 8);
                o[0] = f4{part[0], part[1], part[2], part[3]};
                o[1] = f4{part[4], part[5], part[6], part[7]};
            }
        }
        if (last_step && ng * 8 < D) {
            const int64_t d = ng * 8 + lane;
            float part = 0.0f;
            for (int u = 0; u < cnt; ++u) {
                const int64_t row_at = __builtin_amdgcn_readlane(e.pos, l + u);
                if (d < D) part = part + grad_elem(grad[row_at * D + d], scale, scale_mode);
            }
            if (d < D) {
                if (only) out[row * D + d] = finish(0.0f + part, scale, scale_mode);
                else dst[d] = part;
            }
        }
    }
}

// One output row without occurrences, or with at most kDirect: zeros, or all G column groups of a lane (64 groups of 8
// columns apart) of all its occurrences in flight together, the gradient rows coming from HBM.  `at`: their positions.
template <bool FEW, int G, int N>
__device__ __forceinline__ void sum_direct(const int* at, int n, const uint16_t* __restrict__ grad, int64_t D, float scale,
                                           int scale_mode, bool wide, uint16_t* __restrict__ orow) {
    const int lane = threadIdx.x, ng = (int)(D / 8);
    for (int gi = lane; gi < ng; gi += kEmbThreads * G) {
        u4 x[N][G];
#pragma unroll
        for (int u = 0; u < N; ++u)
#pragma unroll
            for (int g = 0; g < G; ++g)
                if (u < n && gi + g * kEmbThreads < ng)
                    x[u][g] = load8(grad + (int64_t)at[u] * D + (gi + g * kEmbThreads) * 8);
#pragma unroll
        for (int g = 0; g < G; ++g) {
            float acc[8], part[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) acc[k] = part[k] = 0.0f;
#pragma unroll
            for (int u = 0; u < N; ++u) {
                if (u < n) {
                    if (FEW && u > 0 && at[u] / kFewRowsChunk != at[u - 1] / kFewRowsChunk) {
#pragma unroll
                        for (int k = 0; k < 8; ++k) {
                            acc[k] = add_part<FEW>(acc[k], part[k]);
                            part[k] = 0.0f;
                        }
                    }
#pragma unroll
                    for (int k = 0; k < 8; ++k) part[k] = part[k] + grad_elem(col(x[u][g], k), scale, scale_mode);
                }
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) acc[k] = add_part<FEW>(acc[k], part[k]);
            const u4 o = finish8(acc, scale, scale_mode);
            if (gi + g * kEmbThreads < ng) row_store8(orow, wide, ng * 16, (gi + g * kEmbThreads) * 16, o);
        }
    }
    const int d = ng * 8 + lane;
    if (d < D) {
        float acc = 0.0f, part = 0.0f;
#pragma unroll
        for (int u = 0; u < N; ++u) {
            if (u < n) {
                if (FEW && u > 0 && at[u] / kFewRowsChunk != at[u - 1] / kFewRowsChunk) {
                    acc = add_part<FEW>(acc, part);
                    part = 0.0f;
                }
                part = part + grad_elem(grad[(int64_t)at[u] * D + d], scale, scale_mode);
            }
        }
        orow[d] = finish(add_part<FEW>(acc, part), scale, scale_mode);
    }
}

// One output row of n <= kDirectDense occurrences, the sorted places from lo on, group by group: the rows of a run (at
// most 10) are loaded together.
__device__ __forceinline__ void sum_row_runs(const Ent* __restrict__ ent, int lo, int n,
                                             const uint16_t* __restrict__ grad, int64_t D, float scale, int scale_mode,
                                             bool wide, uint16_t* __restrict__ orow) {
    const int lane = threadIdx.x, ng = (int)(D / 8);
    const int pos = lane < n ? ent[lo + lane].pos : 0;
    int at[kDirectDense];
#pragma unroll
    for (int u = 0; u < kDirectDense; ++u) at[u] = __builtin_amdgcn_readlane(pos, u);
    for (int gi = lane; gi < ng; gi += kEmbThreads) {
        float acc[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) acc[k] = 0.0f;
#pragma unroll
        for (int k0 = 0; k0 < kDirectDense; k0 += kRowsPerPartial) {
            if (k0 < n) {
                u4 x[kRowsPerPartial];
#pragma unroll
                for (int u = 0; u < kRowsPerPartial; ++u)
                    if (k0 + u < n) x[u] = load8(grad + (int64_t)at[k0 + u] * D + (int64_t)gi * 8);
                float part[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) part[k] = 0.0f;
#pragma unroll
                for (int u = 0; u < kRowsPerPartial; ++u) {
                    if (k0 + u < n) {
#pragma unroll
                        for (int k = 0; k < 8; ++k) part[k] = part[k] + grad_elem(col(x[u], k), scale, scale_mode);
                    }
                }
#pragma unroll
                for (int k = 0; k < 8; ++k) acc[k] = acc[k] + part[k];
            }
        }
        row_store8(orow, wide, ng * 16, gi * 16, finish8(acc, scale, scale_mode));
    }
    const int d = ng * 8 + lane;
    if (d < D) {
        float acc = 0.0f;
#pragma unroll
        for (int k0 = 0; k0 < kDirectDense; k0 += kRowsPerPartial) {
            if (k0 < n) {
                float part = 0.0f;
#pragma unroll
                for (int u = 0; u < kRowsPerPartial; ++u)
                    if (k0 + u < n) part = part + grad_elem(grad[(int64_t)at[k0 + u] * D + d], scale, scale_mode);
                acc = acc + part;
            }
        }
        orow[d] = finish(acc, scale, scale_mode);
    }
}

// Workgroups [0, run_waves): runs of ids of more than kDirect occurrences (DENSE: kDirectDense); then one per output row,
// which writes it unless the runs do.
template <bool FEW, int G, bool DENSE>
__global__ __launch_bounds__(kEmbThreads) void emb_rows_kernel(const uint16_t* __restrict__ grad, int64_t D, int64_t V,
                                                               const Ent* __restrict__ ent,
                                                               const int2* __restrict__ info, int64_t padding_idx,
                                                               float scale, int scale_mode, uint16_t* __restrict__ out,
                                                               int run_waves, int steps, int block,
                                                               int* __restrict__ counts,
                                                               int32_t* __restrict__ short_list,
                                                               int32_t* __restrict__ long_list,
                                                               float* __restrict__ parts) {
    if ((int)blockIdx.x < run_waves) {
        const int b = (int)blockIdx.x;
        const int step = b % steps, run_block = DENSE ? block : FEW ? kFewBlock : kRunBlock;
        const int64_t valid = counts[2];
        for (int64_t p0 = (int64_t)(b / steps) * run_block; p0 < valid; p0 += (int64_t)(run_waves / steps) * run_block)
            sum_runs<FEW, DENSE ? kDirectDense : kDirect>(p0, run_block, step, step == steps - 1, grad, D, ent, padding_idx,
                                                          scale, scale_mode, valid, out, counts, short_list, long_list,
                                                          parts);
        return;
    }
    // Row of workgroup b (run_waves is a multiple of 8: workgroup b runs on XCD b mod 8): each XCD takes kSpan consecutive
    // rows of every 8 kSpan.  (More rows than kMaxRowWaves: in several rounds.)
    const int lane = threadIdx.x, ng = (int)(D / 8);
    const bool wide = D % 8 == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
    for (int64_t b = blockIdx.x - run_waves; b < V + 8 * kSpan; b += gridDim.x - run_waves) {
        const int64_t t = (b & ~(int64_t)(8 * kSpan - 1)) + (b & 7) * kSpan + ((b >> 3) & (kSpan - 1));
        if (t >= V) continue;
        const int2 r = info[t];
        uint16_t* orow = out + t * D;
        if (r.y == 0 || t == padding_idx) {
            for (int gi = lane; gi < ng; gi += kEmbThreads) row_store8(orow, wide, ng * 16, gi * 16, u4{0u, 0u, 0u, 0u});
            if (ng * 8 + lane < D) orow[ng * 8 + lane] = 0;
        } else if (r.y == 1) {
            const int at[1] = {r.x};
            sum_direct<FEW, G, 1>(at, 1, grad, D, scale, scale_mode, wide, orow);
        } else if (r.y <= kDirect) {
            const int pos = lane < r.y ? ent[r.x + lane].pos : 0;
            int at[kDirect];
#pragma unroll
            for (int u = 0; u < kDirect; ++u) at[u] = __builtin_amdgcn_readlane(pos, u);
            sum_direct<FEW, G, kDirect>(at, r.y, grad, D, scale, scale_mode, wide, orow);
        } else if (DENSE && r.y <= kDirectDense) {
            sum_row_runs(ent, r.x, r.y, grad, D, scale, scale_mode, wide, orow);
        }
    }
}

// The sum of n partials of one column in LDS rows 0 .. n - 1, added in order to acc, 16 reads in flight.  The adds of a
// whole 16 follow each other at their own latency; with a choice after each the chain launch of 65,536 Zipf ids of width
// 256 into 256 rows took 28.2 us, without 21.2 (50,000 of 64 into 8000 rows 21.6 / 16.4, few indices 15.4 / 14.0).
template <bool FEW>
__device__ __forceinline__ float chain_rows(float acc, const float (*buf)[kWave], int n, int lane) {
    int k0 = 0;
    for (; k0 + 16 <= n; k0 += 16) {
        float y[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) y[i] = buf[k0 + i][lane];
#pragma unroll
        for (int i = 0; i < 16; ++i) acc = add_part<FEW>(acc, y[i]);
    }
    if (k0 < n) {
        float y[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) y[i] = buf[k0 + i][lane];
#pragma unroll
        for (int i = 0; i < 16; ++i)
            if (k0 + i < n) acc = add_part<FEW>(acc, y[i]);
    }
    return acc;
}

// The ids of several runs: each (id, 64 columns) is an item, one column per lane, whose run partials are added in run
// order -- aten's order -- and rounded to the bf16 row.
//   - ids of more than kWaveChainRuns runs (long_list): workgroup g takes the items g, g + G, ...; per batch its waves
//     load the id's next kChainRows partials into LDS (kChainDepth loads in flight per lane), then wave 0 adds them to
//     its accumulator;
//   - the others (short_list): wave w of the grid takes the items w, w + W, ..., loads all of the id's partials at once
//     and adds them in registers, with no barrier.
// The lists hold the ids' first sorted places.
__global__ __launch_bounds__(kWave * kChainWaves) void emb_chain_kernel(const float* __restrict__ parts, int64_t D,
                                                                       const Ent* __restrict__ ent,
                                                                       const int32_t* __restrict__ short_list,
                                                                       const int32_t* __restrict__ long_list,
                                                                       const int* __restrict__ counts, float scale,
                                                                       int scale_mode, uint16_t* __restrict__ out) {
    __shared__ float buf[kChainRows][kWave];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
    const int64_t ncg = (D + kWave - 1) / kWave;
    const int64_t long_items = (int64_t)counts[1] * ncg;
    for (int64_t item = blockIdx.x; item < long_items; item += gridDim.x) {
        const int64_t c = (item % ncg) * kWave + lane;
        const bool valid = c < D;
        const Ent e = ent[long_list[item / ncg]];
        const int64_t nrun = ((int64_t)e.n + kRowsPerPartial - 1) / kRowsPerPartial;
        const float* src = parts + run_slot<false>(e.lo, e.lo) * D + c;
        float acc = 0.0f;
        for (int64_t b = 0; b < nrun; b += kChainRows) {
            float x[kChainDepth];
#pragma unroll
            for (int i = 0; i < kChainDepth; ++i) {
                const int64_t k = b + wave + (int64_t)kChainWaves * i;
                x[i] = (k < nrun && valid) ? src[k * D] : 0.0f;
            }
#pragma unroll
            for (int i = 0; i < kChainDepth; ++i) buf[wave + kChainWaves * i][lane] = x[i];
            __syncthreads();
            if (wave == 0) acc = chain_rows<false>(acc, buf, (int)(nrun - b < kChainRows ? nrun - b : kChainRows), lane);
            __syncthreads();
        }
        if (wave == 0 && valid) out[(int64_t)e.id * D + c] = finish(acc, scale, scale_mode);
    }
    const int64_t items = (int64_t)counts[0] * ncg;
    for (int64_t item = (int64_t)blockIdx.x * kChainWaves + wave; item < items;
         item += (int64_t)gridDim.x * kChainWaves) {
        const int64_t c = (item % ncg) * kWave + lane;
        if (c >= D) continue;
        const Ent e = ent[short_list[item / ncg]];
        const int nrun = (e.n + kRowsPerPartial - 1) / kRowsPerPartial;
        const float* src = parts + run_slot<false>(e.lo, e.lo) * D + c;
        float x[kWaveChainRuns];
#pragma unroll
        for (int k = 0; k < kWaveChainRuns; ++k) x[k] = k < nrun ? src[(int64_t)k * D] : 0.0f;
        float acc = 0.0f;
#pragma unroll
        for (int k = 0; k < kWaveChainRuns; ++k)
            if (k < nrun) acc = acc + x[k];
        out[(int64_t)e.id * D + c] = finish(acc, scale, scale_mode);
    }
}

// The same for few indices, where any occurrence may start a run, and an id has at most kFewRuns of them.
//   - ids of more than kWaveChainRuns occurrences: the workgroup first lists their runs in LDS (each wave finds the
//     starts among 64 places at a time, its first one's number is the runs of the waves and rounds before it), loads all
//     of the partials, and wave 0 adds them;
//   - the others: one wave's lanes find the starts.
__global__ __launch_bounds__(kWave * kChainWaves) void emb_chain_few_kernel(const float* __restrict__ parts, int64_t D,
                                                                           const Ent* __restrict__ ent,
                                                                           const int32_t* __restrict__ short_list,
                                                                           const int32_t* __restrict__ long_list,
                                                                           const int* __restrict__ counts, float scale,
                                                                           int scale_mode, uint16_t* __restrict__ out) {
    __shared__ float buf[kFewRuns][kWave];
    __shared__ int run[kFewRuns], found[kChainWaves];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
    const int64_t ncg = (D + kWave - 1) / kWave;
    auto starts_at = [&](const Ent& e, int p) {
        return p < e.lo + e.n && run_starts<true>(p, e.lo, ent[p].pos, p > e.lo ? ent[p - 1].pos : 0);
    };
    const int64_t long_items = (int64_t)counts[1] * ncg;
    for (int64_t item = blockIdx.x; item < long_items; item += gridDim.x) {
        const int64_t c = (item % ncg) * kWave + lane;
        const bool valid = c < D;
        const Ent e = ent[long_list[item / ncg]];
        int nrun = 0;
        for (int b = 0; b < e.n; b += kWave * kChainWaves) {
            const int p = e.lo + b + (int)threadIdx.x;
            const uint64_t m = __ballot(starts_at(e, p));
            if (lane == 0) found[wave] = __builtin_popcountll(m);
            __syncthreads();
            int at = nrun;
            for (int w = 0; w < kChainWaves; ++w) {
                at += w < wave ? found[w] : 0;
                nrun += found[w];
            }
            if (m >> lane & 1) run[at + __builtin_popcountll(m & ((1ull << lane) - 1))] = p;
            __syncthreads();
        }
        constexpr int kDepth = kFewRuns / kChainWaves;
        float x[kDepth];
#pragma unroll
        for (int i = 0; i < kDepth; ++i) {
            const int k = wave + kChainWaves * i;
            x[i] = (k < nrun && valid) ? parts[(int64_t)run[k < nrun ? k : 0] * D + c] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < kDepth; ++i) buf[wave + kChainWaves * i][lane] = x[i];
        __syncthreads();
        if (wave == 0 && valid)
            out[(int64_t)e.id * D + c] = finish(chain_rows<true>(0.0f, buf, nrun, lane), scale, scale_mode);
        __syncthreads();
    }
    const int64_t items = (int64_t)counts[0] * ncg;
    for (int64_t item = (int64_t)blockIdx.x * kChainWaves + wave; item < items;
         item += (int64_t)gridDim.x * kChainWaves) {
        const int64_t c = (item % ncg) * kWave + lane;
        const Ent e = ent[short_list[item / ncg]];
        const uint64_t m = __ballot(starts_at(e, e.lo + lane));
        const float* src = parts + (int64_t)e.lo * D + c;
        float x[kWaveChainRuns];
#pragma unroll
        for (int k = 0; k < kWaveChainRuns; ++k) x[k] = (m >> k & 1) && c < D ? src[(int64_t)k * D] : 0.0f;
        float acc = 0.0f;
#pragma unroll
        for (int k = 0; k < kWaveChainRuns; ++k)
            if (m >> k & 1) acc = add_part<true>(acc, x[k]);
        if (c < D) out[(int64_t)e.id * D + c] = finish(acc, scale, scale_mode);
    }
}

// Stable sort of the (key, position) pairs by key: equal keys keep their position order, which is aten's order.
// end_bit bounds the radix sort's passes (keys are at most V); merge selects the sort that records no memset.
hipError_t sort_pairs(void* temp, size_t& bytes, const uint32_t* keys, uint32_t* skeys, const int32_t* vals,
                      int32_t* svals, int64_t R, int end_bit, bool merge, hipStream_t st) {
    if (merge)
        return rocprim::merge_sort(temp, bytes, keys, skeys, vals, svals, (size_t)R, rocprim::less<uint32_t>(), st);
    return hipcub::DeviceRadixSort::SortPairs(temp, bytes, keys, skeys, vals, svals, (int)R, 0, end_bit, st);
}

size_t sort_temp_bytes(int64_t R) {
    size_t radix = 0, merge = 0;
    (void)sort_pairs(nullptr, radix, nullptr, nullptr, nullptr, nullptr, R, 32, false, 0);
    (void)sort_pairs(nullptr, merge, nullptr, nullptr, nullptr, nullptr, R, 32, true, 0);
    return radix > merge ? radix : merge;
}

// Whether work enqueued on `st` is being captured into a graph (an error reads as not capturing).
bool capturing(hipStream_t st) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(st, &status) == hipSuccess && status != hipStreamCaptureStatusNone;
}

inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// Whether the occurrences are put in order by emb_bucket_kernel (else by the library sort).
bool bucketed(int64_t R, int64_t V) { return R <= kBucketRows && V <= kBucketVocab; }

// Workspace: ent (R), info (V), the three counters (ids in short_list and in long_list, ids inside the vocabulary), the
// two lists (ids of at least 11 occurrences, of more than kDirect for few indices), the fp32 partials (R / 4 slots, R for
// few indices, D each), then, for the library sort, its keys and positions and their sorted copies (R each) and its
// temporary storage.
struct EmbWorkspace {
    Ent* ent;
    int2* info;
    int* counts;
    int32_t* short_list;
    int32_t* long_list;
    float* parts;
    uint32_t* keys;
    int32_t* vals;
    uint32_t* skeys;
    int32_t* svals;
    void* temp;
    size_t temp_bytes;
    size_t total;
};

EmbWorkspace emb_workspace(void* base, int64_t R, int64_t D, int64_t V) {
    EmbWorkspace w{};
    unsigned char* p = static_cast<unsigned char*>(base);
    size_t off = 0;
    auto take = [&](size_t bytes) {
        unsigned char* q = p ? p + off : nullptr;
        off += align256(bytes > 0 ? bytes : 1);
        return q;
    };
    const bool few = R < kSortMinRows;
    const size_t r = (size_t)R, listed = r / (few ? kDirect + 1 : kRowsPerPartial + 1);
    const size_t slots = few ? r : r / kSlotSpan + 1;
    w.ent = reinterpret_cast<Ent*>(take(sizeof(Ent) * r));
    w.info = reinterpret_cast<int2*>(take(sizeof(int2) * (size_t)V));
    w.counts = reinterpret_cast<int*>(take(3 * sizeof(int)));
    w.short_list = reinterpret_cast<int32_t*>(take(sizeof(int32_t) * listed));
    w.long_list = reinterpret_cast<int32_t*>(take(sizeof(int32_t) * listed));
    w.parts = reinterpret_cast<float*>(take(sizeof(float) * slots * (size_t)D));
    if (!bucketed(R, V)) {
        w.keys = reinterpret_cast<uint32_t*>(take(sizeof(uint32_t) * r));
        w.vals = reinterpret_cast<int32_t*>(take(sizeof(int32_t) * r));
        w.skeys = reinterpret_cast<uint32_t*>(take(sizeof(uint32_t) * r));
        w.svals = reinterpret_cast<int32_t*>(take(sizeof(int32_t) * r));
        w.temp_bytes = sort_temp_bytes(R);
        w.temp = take(w.temp_bytes);
    }
    w.total = off;
    return w;
}

bool dense(int64_t R, int64_t V) { return R >= kDenseRows && R >= kDenseMean * V; }

struct RowsCall {
    const uint16_t* grad;
    int64_t R, D, V, padding_idx;
    float scale;
    int scale_mode;
    uint16_t* out;
    size_t lds;
    hipStream_t st;
};

// The rows launch, with as many column groups per lane as the row needs, at most 6 (D 3072).
template <bool FEW, int G, bool DENSE = false>
void launch_rows_g(const RowsCall& c, const EmbWorkspace& w) {
    const int64_t steps = (c.D / 8 + kEmbThreads - 1) / kEmbThreads, step_waves = steps > 0 ? steps : 1;
    int64_t run_waves = 0;
    int block = FEW ? kFewBlock : kRunBlock;
    if (c.R > kDirect) {
        if (DENSE && c.R >= kShortBlockMean * c.V)
            block = c.R * step_waves <= kQuarterWaves * (kRunBlock / 2) ? kRunBlock / 4 : kRunBlock / 2;
        const int64_t blocks = (c.R + block - 1) / block, most = kMaxWaves / step_waves;      // steps <= 32,768
        run_waves = ((blocks < most ? blocks : most) + 7) / 8 * 8 * step_waves;
    }
    const int64_t spans = (c.V + 8 * kSpan - 1) / (8 * kSpan) * (8 * kSpan);
    const int64_t rows = spans < kMaxRowWaves ? spans : kMaxRowWaves;
    hipLaunchKernelGGL((emb_rows_kernel<FEW, G, DENSE>), dim3((unsigned)(run_waves + rows)), dim3(kEmbThreads), c.lds, c.st,
                       c.grad, c.D, c.V, w.ent, w.info, c.padding_idx, c.scale, c.scale_mode, c.out, (int)run_waves,
                       (int)step_waves, block, w.counts, w.short_list, w.long_list, w.parts);
}

template <bool FEW>
void launch_rows(const RowsCall& c, const EmbWorkspace& w) {
    const int64_t need = (c.D / 8 + kEmbThreads - 1) / kEmbThreads;          // groups per lane
    const int64_t steps = (need + 5) / 6;
    switch (need > 0 ? (need + steps - 1) / steps : 1) {
        case 1: return launch_rows_g<FEW, 1>(c, w);
        case 2: return launch_rows_g<FEW, 2>(c, w);
        case 3: return launch_rows_g<FEW, 3>(c, w);
        case 4: return launch_rows_g<FEW, 4>(c, w);
        case 5: return launch_rows_g<FEW, 5>(c, w);
        default: return launch_rows_g<FEW, 6>(c, w);
    }
}

}  // namespace

extern "C" {

int64_t z1_embedding_backward_workspace(int64_t R, int64_t D, int64_t V) {
    if (R < 0 || R > INT32_MAX || D <= 0 || D > kMaxCols || V <= 0 || V > INT32_MAX - 1) return Z1_E_SIZE;
    return (int64_t)emb_workspace(nullptr, R, D, V).total;
}

int z1_embedding_backward(const int64_t* ids, const uint16_t* grad, int64_t R, int64_t D, int64_t V,
                          int64_t padding_idx, float scale, int scale_mode, uint16_t* out, void* workspace,
                          int64_t workspace_bytes, void* stream) {
    if (!out || !workspace || (R > 0 && (!ids || !grad))) return Z1_E_NULL;
    if (scale_mode < 0 || scale_mode > 2) return Z1_E_MODE;
    const int64_t need = z1_embedding_backward_workspace(R, D, V);
    if (need < 0) return (int)need;
    if (workspace_bytes < need) return Z1_E_WORKSPACE;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const EmbWorkspace w = emb_workspace(workspace, R, D, V);
    hipError_t e = hipSuccess;
    if (bucketed(R, V)) {
        int kb = kMinBucketBits;
        while ((((V - 1) >> (kGranuleBits + kb)) + 1) << kGranuleBits > kMaxLocal / 2 && kb < kMaxBucketBits) ++kb;
        hipLaunchKernelGGL(emb_bucket_kernel, dim3(1u << kb), dim3(kBucketThreads), 0, st, ids, (int)R, (int)V, kb, w.ent,
                           w.info, w.counts);
    } else {
        const dim3 per_row((unsigned)((R + 255) / 256));
        if (R > 0) {
            hipLaunchKernelGGL(emb_keys_kernel, per_row, dim3(256), 0, st, ids, R, V, w.keys, w.vals);
            e = hipGetLastError();
            if (e != hipSuccess) return (int)e;
            size_t tb = w.temp_bytes;
            int end_bit = 1;
            while (end_bit < 32 && ((uint64_t)V >> end_bit) != 0) ++end_bit;   // keys are <= V
            e = sort_pairs(w.temp, tb, w.keys, w.skeys, w.vals, w.svals, R, end_bit, capturing(st), st);
            if (e != hipSuccess) return (int)e;
        }
        const int64_t vocab_blocks = (V + kPlaceThreads - 1) / kPlaceThreads, blocks = (R + kPlaceThreads - 1) / kPlaceThreads;
        const bool search = R <= kSearchRows;
        hipLaunchKernelGGL(emb_places_kernel, dim3((unsigned)(vocab_blocks + (search ? blocks : 0))), dim3(kPlaceThreads), 0,
                           st, w.skeys, w.svals, R, V, (int)vocab_blocks, w.info, w.ent, w.counts);
        e = hipGetLastError();
        if (e != hipSuccess) return (int)e;
        if (!search)
            hipLaunchKernelGGL(emb_entries_kernel, dim3((unsigned)blocks), dim3(kPlaceThreads), 0, st, w.skeys, w.svals, R, V,
                               w.info, w.ent);
    }
    e = hipGetLastError();
    if (e != hipSuccess) return (int)e;
    int dev = 0;
    e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    RowsCall c{grad, R, D, V, padding_idx, scale, scale_mode, out, 0, st};
    const bool few = R < kSortMinRows;                  // aten's kernel for few indices: its order
    if (dense(R, V)) {
        launch_rows_g<false, 1, true>(c, w);
    } else {
        const int rc = z1detail::occupancy_lds(dev, kEmbWgPerCu, &c.lds);
        if (rc) return rc;
        if (few) launch_rows<true>(c, w);
        else launch_rows<false>(c, w);
    }
    e = hipGetLastError();
    if (e != hipSuccess) return (int)e;
    // the most items the lists can hold
    const int64_t items = R / (few ? kDirect + 1 : kRowsPerPartial + 1) * ((D + kWave - 1) / kWave);
    if (items == 0) return Z1_OK;
    const dim3 grid((unsigned)(items < kChainGrid ? items : kChainGrid)), threads(kWave * kChainWaves);
    if (few)
        hipLaunchKernelGGL(emb_chain_few_kernel, grid, threads, 0, st, w.parts, D, w.ent, w.short_list, w.long_list,
                           w.counts, scale, scale_mode, out);
    else
        hipLaunchKernelGGL(emb_chain_kernel, grid, threads, 0, st, w.parts, D, w.ent, w.short_list, w.long_list, w.counts,
                           scale, scale_mode, out);
    return (int)hipGetLastError();
}

}  // extern "C"
