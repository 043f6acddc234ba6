// yoco_z1: the owner's token-embedding gradient (declarations: include/yoco_z1.h).
//
// Replaces torch.ops.aten.embedding_dense_backward(g_all, ids, V, padding_idx, False) on the embedding's owner,
// followed or preceded by the x 1/world of the reference (yoco/models/decoder/layer_graphs.py:87-93,
// yoco/models/decoder/ce_reduce.py:226-231).  Same summation order as aten for the row count.  For more than 3072
// indices aten sorts: occurrences of each token id in stable position order, fp32 partial sums over runs of 10
// consecutive occurrences, the partials summed in order, one rounding to bf16.  For fewer its other kernel walks
// the indices in chunks of 16: per chunk and id an fp32 sum in position order, rounded to bf16 and added to the
// bf16 row (emb_rows_kernel<true>; no heavy passes).  padding_idx rows and ids outside [0, V) contribute nothing.
//
//   1. each id's occurrences in position order (spos) and where they are (rng[t] = first sorted position, count): for
//      up to kBucketRows rows one launch, emb_bucket_kernel; beyond, keys[i] = id_i (or V when out of range) and
//      vals[i] = i sorted stably by key -- hipCUB's radix sort, or, while the stream is being captured into a HIP
//      graph, rocPRIM's merge sort, which clears nothing with memsets (the radix sort does; both are stable, so the
//      order is the same) -- and one binary search per t over the sorted keys;
//   2. one wave per output row t writes the row's sums -- or zeros -- exactly once, 8 bf16 columns per lane and
//      group, with nontemporal stores (aten zero-fills the whole table and then scatters into it; here every row of
//      the table is written once), for ids with at most kHeavyRows occurrences; the others are listed, with a slot
//      range for their runs, for
//   3. emb_heavy_parts_kernel, which forms every run partial of every heavy id in parallel over the whole chip
//      into an fp32 workspace, and
//   4. emb_heavy_chain_kernel, which adds each heavy id's partials in run order per column.  Token frequencies in
//      text are skewed: one wave (or one workgroup) walking thousands of occurrences of one id would take
//      milliseconds.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>
#include <rocprim/device/device_merge_sort.hpp>

#include <stdint.h>

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
// resident row workgroups per CU, capped with a dynamic LDS reservation the kernel does not use: 0.131 ms per call
// at 9-10 per CU against 0.148 ms at the 32 the waves allow (0.144 at 16, 0.136 at 8, 0.146 at 7, 0.180 at 6)
constexpr int kEmbWgPerCu = 10;
constexpr int kWave = 64;
// tokens with more occurrences go to the heavy passes; a heavy token's ceil(n / 10) runs are at most n / 7 for
// n >= 21, so the run slots of all heavy tokens number at most R / 7
constexpr int kHeavyRows = 20;
static_assert(kHeavyRows >= 20, "the run-slot bound R / 7 needs heavy tokens of at least 21 occurrences");
constexpr int kPartsThreads = 256;         // heavy pass 1: one run x column group per wave
constexpr int kPartsGrid = 2048;
constexpr int kChainWaves = 16;            // heavy pass 2: waves that load a batch of partials
constexpr int kChainDepth = 16;            // partials per lane per batch
constexpr int kChainRows = kChainWaves * kChainDepth;
static_assert(kChainRows % 16 == 0, "wave 0 reads a batch 16 rows at a time");
constexpr int kChainGrid = 512;
constexpr int kWaveChainRuns = 32;         // heavy tokens of at most this many runs are chained by one wave
constexpr int64_t kMaxCols = 1 << 24;      // D limit: keeps the workspace size and offsets far from overflow

__device__ __forceinline__ float bf16f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

__device__ __forceinline__ uint16_t bf16r(float x) {
    const uint32_t u = __float_as_uint(x);
    if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0u;
    return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

__global__ void emb_keys_kernel(const int64_t* __restrict__ ids, int64_t R, int64_t V, uint32_t* __restrict__ keys,
                                int32_t* __restrict__ vals) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= R) return;
    const int64_t t = ids[i];
    keys[i] = (t >= 0 && t < V) ? (uint32_t)t : (uint32_t)V;
    vals[i] = (int32_t)i;
}

// rng[t] = (first index of the sorted keys that is >= t, number of keys equal to t), for t in [0, V).  Independent
// binary searches, one thread per t (the latency of the searches overlaps).
__global__ void emb_row_ranges_kernel(const uint32_t* __restrict__ sorted, int64_t R, int64_t V,
                                      int2* __restrict__ rng, int* __restrict__ counts) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t == 0) {                               // the rows kernel appends the heavy tokens after this kernel
        counts[0] = 0;
        counts[1] = 0;
        counts[2] = 0;
    }
    if (t >= V) return;
    auto lower = [&](uint32_t key) {
        int64_t lo = 0, hi = R;
        while (lo < hi) {
            const int64_t mid = (lo + hi) >> 1;
            if (sorted[mid] < key) lo = mid + 1;
            else hi = mid;
        }
        return (int32_t)lo;
    };
    const int32_t lo = lower((uint32_t)t);
    rng[t] = int2{lo, lower((uint32_t)t + 1) - lo};
}

// The same results (spos, the sorted keys and rng) in one launch, without a sort over the whole list.  The ids are
// split over 2^kb buckets, granules of 2^kGranuleBits consecutive ids round robin, one workgroup per bucket (text's
// frequent ids are the small ones: spread, no workgroup gets them all).  Every workgroup reads all R ids, wave w the
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
// 80 us at 16,384 rows), single ids scatter rng in 8-byte writes (52 / 71 us); fewer than 2^8 buckets leave
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

__global__ __launch_bounds__(kBucketThreads) void emb_bucket_kernel(const int64_t* __restrict__ ids, int R, int V,
                                                                    int kb, int32_t* __restrict__ spos,
                                                                    uint32_t* __restrict__ skeys,
                                                                    int2* __restrict__ rng, int* __restrict__ counts) {
    __shared__ int hist[kBucketWaves][kMaxLocal];
    __shared__ int wsum[kBucketWaves], wless[kBucketWaves];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
    const int k = blockIdx.x, mask = (1 << kb) - 1;
    if (k == 0 && threadIdx.x < 3) counts[threadIdx.x] = 0;   // the rows kernel appends the heavy tokens after this
    for (int i = lane; i < kMaxLocal; i += kWave) hist[wave][i] = 0;        // this wave's own counters
    // a wave's segment: positions [s0, s1), 64 consecutive ones a step
    const int steps = (R + kBucketThreads - 1) / kBucketThreads;
    const int s0 = wave * steps * kWave, s1 = s0 + steps * kWave < R ? s0 + steps * kWave : R;
    int loc[kBucketTile];                    // local id, -1: another bucket's (or out of range)
    int less = 0;
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
            const bool ok = t[i] >= 0 && t[i] < V;
            const int id = (int)t[i], b = (id >> kGranuleBits) & mask;
            loc[i] = ok && b == k ? ((id >> (kGranuleBits + kb)) << kGranuleBits) | (id & ((1 << kGranuleBits) - 1)) : -1;
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
    if (l < kMaxLocal) {
#pragma unroll
        for (int w = 0; w < kBucketWaves; ++w) hist[w][l] += start;
        const int64_t t = ((int64_t)(l >> kGranuleBits) << (kGranuleBits + kb)) + ((int64_t)k << kGranuleBits) +
                          (l & ((1 << kGranuleBits) - 1));
        if (t < V) rng[t] = int2{start, cnt};
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
                if (mine) {
                    const int pos = at + __builtin_popcountll(same & ((1ull << lane) - 1));
                    spos[pos] = p0 + i * kWave + lane;
                    skeys[pos] = (uint32_t)(((l0 >> kGranuleBits) << (kGranuleBits + kb)) + (k << kGranuleBits) +
                                            (l0 & ((1 << kGranuleBits) - 1)));
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
// (layer_graphs.py:93).
__device__ __forceinline__ uint16_t finish(float acc, float scale, int scale_mode) {
    uint16_t o = bf16r(acc);
    if (scale_mode == 2) o = bf16r(bf16f(o) * scale);
    return o;
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

// Adds a finished partial to the row's sum: aten's sort path adds fp32 partials; its few-indices kernel rounds the
// partial to bf16 and the row after the add.
template <bool FEW>
__device__ __forceinline__ float add_part(float acc, float part) {
    return FEW ? bf16f(bf16r(acc + bf16f(bf16r(part)))) : acc + part;
}

// Whether occurrence j of a row whose occurrences start at lo begins another partial (j > lo): every 10th occurrence,
// or, for few indices, where the next chunk of 16 indices begins.
template <bool FEW>
__device__ __forceinline__ bool new_part(const int32_t* __restrict__ spos, int64_t lo, int64_t j) {
    return FEW ? spos[j] / kFewRowsChunk != spos[j - 1] / kFewRowsChunk : (j - lo) % kRowsPerPartial == 0;
}

// A row with one occurrence: all G of a lane's column groups (gi, gi + 64, ... below ng, 8 columns each) loaded at once
// -- the gradient row comes from HBM, so the wave waits for memory once a row instead of once a group -- and rounded.
// With this and sum_row below, 16,384 rows of 3072 into a 100,288-row table, gradients not in a cache: 163 us a call
// against 205 us with each group loaded, summed and stored before the next (Zipf ids 205 against 231 us).
template <int G>
__device__ __forceinline__ void copy_row(const uint16_t* __restrict__ row, int64_t gi, int64_t ng, float scale,
                                         int scale_mode, uint16_t* __restrict__ orow) {
    u4 x[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        x[g] = u4{0u, 0u, 0u, 0u};
        if (gi + g * kEmbThreads < ng) x[g] = load8(row + (gi + g * kEmbThreads) * 8);
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
        u4 o;
#pragma unroll
        for (int k = 0; k < 4; ++k)       // 0 + x: the sum of one element (-0 gives +0)
            o[k] = (uint32_t)finish(0.0f + grad_elem((uint16_t)x[g][k], scale, scale_mode), scale, scale_mode) |
                   ((uint32_t)finish(0.0f + grad_elem((uint16_t)(x[g][k] >> 16), scale, scale_mode), scale, scale_mode)
                    << 16);
        if (gi + g * kEmbThreads < ng) nt_store8(orow + (gi + g * kEmbThreads) * 8, o);
    }
}

// One row's sum over its occurrences [lo, hi) for G column groups of a lane, as in copy_row: all G loads of an
// occurrence are in flight together, the next occurrence's as well.
template <bool FEW, int G>
__device__ __forceinline__ void sum_row(const uint16_t* __restrict__ grad, int64_t D, const int32_t* __restrict__ spos,
                                        int64_t lo, int64_t hi, int64_t gi, int64_t ng, float scale, int scale_mode,
                                        uint16_t* __restrict__ orow) {
    u4 x[G], y[G];
    float acc[G][8], part[G][8];
    auto load = [&](u4* d, int64_t j) {
        const uint16_t* row = grad + (int64_t)spos[j] * D;
#pragma unroll
        for (int g = 0; g < G; ++g)
            if (gi + g * kEmbThreads < ng) d[g] = load8(row + (gi + g * kEmbThreads) * 8);
    };
#pragma unroll
    for (int g = 0; g < G; ++g) {
        x[g] = y[g] = u4{0u, 0u, 0u, 0u};
#pragma unroll
        for (int k = 0; k < 8; ++k) acc[g][k] = part[g][k] = 0.0f;
    }
    load(x, lo);
    for (int64_t j = lo; j < hi; ++j) {
        if (j + 1 < hi) load(y, j + 1);
        if (j > lo && new_part<FEW>(spos, lo, j)) {
#pragma unroll
            for (int g = 0; g < G; ++g)
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    acc[g][k] = add_part<FEW>(acc[g][k], part[g][k]);
                    part[g][k] = 0.0f;
                }
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
#pragma unroll
            for (int k = 0; k < 8; ++k)
                part[g][k] = part[g][k] + grad_elem((uint16_t)(x[g][k >> 1] >> ((k & 1) * 16)), scale, scale_mode);
            x[g] = y[g];
        }
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
        u4 o;
#pragma unroll
        for (int k = 0; k < 8; k += 2)
            o[k >> 1] = (uint32_t)finish(add_part<FEW>(acc[g][k], part[g][k]), scale, scale_mode) |
                        ((uint32_t)finish(add_part<FEW>(acc[g][k + 1], part[g][k + 1]), scale, scale_mode) << 16);
        if (gi + g * kEmbThreads < ng) nt_store8(orow + (gi + g * kEmbThreads) * 8, o);
    }
}

// One wave per output row t (light tokens: at most kHeavyRows occurrences, and empty or padding rows): the row's
// sums -- or zeros -- written once, G groups of 8 bf16 columns per lane and step, the last D % 8 columns one per lane.
// A token with more occurrences is appended, with the first of its nrun run slots (from counts[1]), to the list of
// tokens of at most kWaveChainRuns runs (heavy_list / heavy_base, count counts[0]) or to that of longer ones
// (long_list / long_base, counts[2]); run_start[slot] = the sorted position of the run's first row.  Its row is left to
// the heavy passes.  The atomics only decide where a token's partials are kept, not how they are summed.
template <bool FEW, int G>
__global__ __launch_bounds__(kEmbThreads) void emb_rows_kernel(const uint16_t* __restrict__ grad, int64_t D,
                                                               const int32_t* __restrict__ spos,
                                                               const int2* __restrict__ rng,
                                                               int64_t padding_idx, float scale, int scale_mode,
                                                               uint16_t* __restrict__ out,
                                                               int* __restrict__ counts,
                                                               int32_t* __restrict__ heavy_list,
                                                               int32_t* __restrict__ heavy_base,
                                                               int32_t* __restrict__ long_list,
                                                               int32_t* __restrict__ long_base,
                                                               int32_t* __restrict__ run_start) {
    // row of workgroup b: undoes the round-robin dispatch over the 8 XCDs, so each XCD writes one contiguous
    // eighth of the table (0.148 vs 0.153 ms per call for t = b)
    int64_t t;
    {
        const int64_t b = blockIdx.x, nb = gridDim.x;
        const int64_t x = b & 7, q = b >> 3, Q = nb >> 3, R = nb & 7;
        t = x * Q + (x < R ? x : R) + q;
    }
    const int lane = threadIdx.x;
    uint16_t* orow = out + t * D;
    const int2 r = rng[t];
    const int64_t lo = r.x, hi = lo + r.y;
    const bool empty = lo == hi || t == padding_idx;
    if (!FEW && !empty && hi - lo > kHeavyRows) {
        const int nrun = (int)((hi - lo + kRowsPerPartial - 1) / kRowsPerPartial);
        int base = 0;
        if (lane == 0) {
            const bool wave_chain = nrun <= kWaveChainRuns;
            const int h = atomicAdd(&counts[wave_chain ? 0 : 2], 1);
            base = atomicAdd(&counts[1], nrun);
            (wave_chain ? heavy_list : long_list)[h] = (int32_t)t;
            (wave_chain ? heavy_base : long_base)[h] = base;
        }
        base = __shfl(base, 0);
        for (int k = lane; k < nrun; k += kEmbThreads) run_start[base + k] = (int32_t)(lo + (int64_t)k * kRowsPerPartial);
        return;
    }
    const int64_t ng = D / 8;
    if (empty) {
        // nontemporal: the 616 MB table is written once and not read back here (0.155 vs 0.184 ms per call)
        for (int64_t gi = lane; gi < ng; gi += kEmbThreads) nt_store8(orow + gi * 8, u4{0u, 0u, 0u, 0u});
    } else {
        // one occurrence (most rows): G groups at a time; more: half as many, whose sums fit the registers that leave
        // room for kEmbWgPerCu resident rows per CU
        constexpr int H = (G + 1) / 2;
        if (hi - lo == 1) {
            const uint16_t* row = grad + (int64_t)spos[lo] * D;
            for (int64_t gi = lane; gi < ng; gi += kEmbThreads * G) copy_row<G>(row, gi, ng, scale, scale_mode, orow);
        } else {
            for (int64_t gi = lane; gi < ng; gi += kEmbThreads * H)
                sum_row<FEW, H>(grad, D, spos, lo, hi, gi, ng, scale, scale_mode, orow);
        }
    }
    const int64_t d = ng * 8 + lane;
    if (d < D) {
        float acc = 0.0f, part = 0.0f;
        for (int64_t j = lo; !empty && j < hi; ++j) {
            if (j > lo && new_part<FEW>(spos, lo, j)) {
                acc = add_part<FEW>(acc, part);
                part = 0.0f;
            }
            part = part + grad_elem(grad[(int64_t)spos[j] * D + d], scale, scale_mode);
        }
        orow[d] = finish(add_part<FEW>(acc, part), scale, scale_mode);
    }
}

// Heavy tokens, pass 1: every run of 10 occurrences of every heavy token, for every column group (512 columns on
// the vector path, 64 otherwise), is one wave's item; the wave sums the run's rows in order (loads issued together)
// and stores the fp32 partial to its run slot of parts (parts[s * D + column]).  The run of slot s starts at sorted
// position run_start[s], and its token is the sorted key there.  Items are spread over the whole
// grid, so one token's thousands of runs are formed in parallel; every wave exits once the items run out.
template <int VEC>
__global__ __launch_bounds__(kPartsThreads) void emb_heavy_parts_kernel(const uint16_t* __restrict__ grad, int64_t D,
                                                                        const int32_t* __restrict__ spos,
                                                                        const uint32_t* __restrict__ skeys,
                                                                        const int2* __restrict__ rng,
                                                                        const int32_t* __restrict__ run_start,
                                                                        const int* __restrict__ counts, float scale,
                                                                        int scale_mode, float* __restrict__ parts) {
    constexpr int kCols = VEC ? 8 : 1;                       // columns per lane
    constexpr int kWaves = kPartsThreads / kWave;
    const int wave = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    const int64_t cols_per_item = (int64_t)kWave * kCols;
    const int64_t ncg = (D + cols_per_item - 1) / cols_per_item;
    const int64_t items = (int64_t)counts[1] * ncg;
    for (int64_t item = (int64_t)blockIdx.x * kWaves + wave; item < items; item += (int64_t)gridDim.x * kWaves) {
        const int64_t s = item / ncg;
        const int64_t c0 = (item % ncg) * cols_per_item + (int64_t)lane * kCols;   // D % 8 == 0 when VEC
        if (c0 >= D) continue;
        const int64_t j0 = run_start[s];
        const int2 r = rng[skeys[j0]];
        const int64_t hi = (int64_t)r.x + r.y;
        const int cnt = (int)(j0 + kRowsPerPartial < hi ? kRowsPerPartial : hi - j0);
        float part[kCols];
#pragma unroll
        for (int k = 0; k < kCols; ++k) part[k] = 0.0f;
        if (VEC) {
            u4 x[kRowsPerPartial];
#pragma unroll
            for (int u = 0; u < kRowsPerPartial; ++u)
                if (u < cnt) x[u] = *reinterpret_cast<const u4*>(grad + (int64_t)spos[j0 + u] * D + c0);
#pragma unroll
            for (int u = 0; u < kRowsPerPartial; ++u) {
                if (u < cnt) {
#pragma unroll
                    for (int k = 0; k < kCols; ++k)
                        part[k] = part[k] + grad_elem((uint16_t)(x[u][k >> 1] >> ((k & 1) * 16)), scale, scale_mode);
                }
            }
        } else {
            uint16_t x[kRowsPerPartial];
#pragma unroll
            for (int u = 0; u < kRowsPerPartial; ++u)
                if (u < cnt) x[u] = grad[(int64_t)spos[j0 + u] * D + c0];
#pragma unroll
            for (int u = 0; u < kRowsPerPartial; ++u)
                if (u < cnt) part[0] = part[0] + grad_elem(x[u], scale, scale_mode);
        }
        float* dst = parts + s * D + c0;
#pragma unroll
        for (int k = 0; k < kCols; ++k) dst[k] = part[k];
    }
}

// Heavy tokens, pass 2: each (heavy token, 64 columns) is an item, one column per lane, whose partials are added in
// run order -- the order of the rows kernel and of aten -- and rounded to the bf16 row.
//   - tokens of more than kWaveChainRuns runs (long_list): workgroup g takes the items g, g + G, ...; per batch its
//     waves load the token's next kChainRows partials into LDS (kChainDepth loads in flight per lane), then wave 0
//     adds them to its accumulator;
//   - the others (heavy_list): wave w of the grid takes the items w, w + W, ..., loads all of the token's partials
//     at once and adds them in registers, with no barrier.
__global__ __launch_bounds__(kWave * kChainWaves) void emb_heavy_chain_kernel(const float* __restrict__ parts,
                                                                             int64_t D,
                                                                             const int2* __restrict__ rng,
                                                                             const int32_t* __restrict__ heavy_list,
                                                                             const int32_t* __restrict__ heavy_base,
                                                                             const int32_t* __restrict__ long_list,
                                                                             const int32_t* __restrict__ long_base,
                                                                             const int* __restrict__ counts,
                                                                             float scale, int scale_mode,
                                                                             uint16_t* __restrict__ out) {
    __shared__ float buf[kChainRows][kWave];
    const int wave = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    const int64_t ncg = (D + kWave - 1) / kWave;
    const int64_t long_items = (int64_t)counts[2] * ncg;
    for (int64_t item = blockIdx.x; item < long_items; item += gridDim.x) {
        const int h = (int)(item / ncg);
        const int64_t col = (item % ncg) * kWave + lane;
        const bool valid = col < D;
        const int64_t t = long_list[h];
        const int64_t nrun = ((int64_t)rng[t].y + kRowsPerPartial - 1) / kRowsPerPartial;
        const float* src = parts + (int64_t)long_base[h] * D + col;
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
            if (wave == 0) {                                   // LDS reads issued 16 at a time, added in order
                const int n = (int)(nrun - b < kChainRows ? nrun - b : kChainRows);
                for (int k0 = 0; k0 < n; k0 += 16) {
                    float y[16];
#pragma unroll
                    for (int i = 0; i < 16; ++i) y[i] = buf[k0 + i][lane];
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        if (k0 + i < n) acc = acc + y[i];
                }
            }
            __syncthreads();
        }
        if (wave == 0 && valid) out[t * D + col] = finish(acc, scale, scale_mode);
    }
    const int64_t items = (int64_t)counts[0] * ncg;
    for (int64_t item = (int64_t)blockIdx.x * kChainWaves + wave; item < items;
         item += (int64_t)gridDim.x * kChainWaves) {
        const int h = (int)(item / ncg);
        const int64_t col = (item % ncg) * kWave + lane;
        if (col >= D) continue;
        const int64_t t = heavy_list[h];
        const int nrun = (rng[t].y + kRowsPerPartial - 1) / kRowsPerPartial;
        const float* src = parts + (int64_t)heavy_base[h] * D + col;
        float x[kWaveChainRuns];
#pragma unroll
        for (int k = 0; k < kWaveChainRuns; ++k) x[k] = k < nrun ? src[(int64_t)k * D] : 0.0f;
        float acc = 0.0f;
#pragma unroll
        for (int k = 0; k < kWaveChainRuns; ++k)
            if (k < nrun) acc = acc + x[k];
        out[t * D + col] = finish(acc, scale, scale_mode);
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

// Workspace: sorted keys and positions (R each), rng (V), the three counters, the two lists of heavy tokens and their
// first run slots (at most R / 21 each), the run starts and the fp32 partials (R / 7 slots, D each), then, for the
// library sort, its keys and positions (R each) and its temporary storage.
struct EmbWorkspace {
    uint32_t* keys;
    int32_t* vals;
    uint32_t* skeys;
    int32_t* svals;
    int2* rng;
    int* counts;
    int32_t* heavy_list;
    int32_t* heavy_base;
    int32_t* long_list;
    int32_t* long_base;
    int32_t* run_start;
    float* parts;
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
    const size_t r = (size_t)R, heavy = (size_t)(R / (kHeavyRows + 1)), slots = (size_t)(R / 7);
    w.skeys = reinterpret_cast<uint32_t*>(take(sizeof(uint32_t) * r));
    w.svals = reinterpret_cast<int32_t*>(take(sizeof(int32_t) * r));
    w.rng = reinterpret_cast<int2*>(take(sizeof(int2) * (size_t)V));
    w.counts = reinterpret_cast<int*>(take(3 * sizeof(int)));
    w.heavy_list = reinterpret_cast<int32_t*>(take(sizeof(int32_t) * heavy));
    w.heavy_base = reinterpret_cast<int32_t*>(take(sizeof(int32_t) * heavy));
    w.long_list = reinterpret_cast<int32_t*>(take(sizeof(int32_t) * heavy));
    w.long_base = reinterpret_cast<int32_t*>(take(sizeof(int32_t) * heavy));
    w.run_start = reinterpret_cast<int32_t*>(take(sizeof(int32_t) * slots));
    w.parts = reinterpret_cast<float*>(take(sizeof(float) * slots * (size_t)D));
    if (!bucketed(R, V)) {
        w.keys = reinterpret_cast<uint32_t*>(take(sizeof(uint32_t) * r));
        w.vals = reinterpret_cast<int32_t*>(take(sizeof(int32_t) * r));
        w.temp_bytes = sort_temp_bytes(R);
        w.temp = take(w.temp_bytes);
    }
    w.total = off;
    return w;
}

// The rows kernel with as many column groups per lane and step as the row needs, at most 6 (D 3072).
template <bool FEW, int G>
void launch_rows_g(int64_t D, int64_t V, size_t lds, hipStream_t st, const uint16_t* grad, const EmbWorkspace& w,
                   int64_t padding_idx, float scale, int scale_mode, uint16_t* out) {
    hipLaunchKernelGGL((emb_rows_kernel<FEW, G>), dim3((unsigned)V), dim3(kEmbThreads), lds, st, grad, D, w.svals,
                       w.rng, padding_idx, scale, scale_mode, out, w.counts, w.heavy_list, w.heavy_base,
                       w.long_list, w.long_base, w.run_start);
}

template <bool FEW>
void launch_rows(int64_t D, int64_t V, size_t lds, hipStream_t st, const uint16_t* grad, const EmbWorkspace& w,
                 int64_t padding_idx, float scale, int scale_mode, uint16_t* out) {
    const int64_t need = (D / 8 + kEmbThreads - 1) / kEmbThreads;          // groups per lane
    const int64_t steps = (need + 5) / 6;
    switch (need > 0 ? (need + steps - 1) / steps : 1) {
        case 1: return launch_rows_g<FEW, 1>(D, V, lds, st, grad, w, padding_idx, scale, scale_mode, out);
        case 2: return launch_rows_g<FEW, 2>(D, V, lds, st, grad, w, padding_idx, scale, scale_mode, out);
        case 3: return launch_rows_g<FEW, 3>(D, V, lds, st, grad, w, padding_idx, scale, scale_mode, out);
        case 4: return launch_rows_g<FEW, 4>(D, V, lds, st, grad, w, padding_idx, scale, scale_mode, out);
        case 5: return launch_rows_g<FEW, 5>(D, V, lds, st, grad, w, padding_idx, scale, scale_mode, out);
        default: return launch_rows_g<FEW, 6>(D, V, lds, st, grad, w, padding_idx, scale, scale_mode, out);
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
        hipLaunchKernelGGL(emb_bucket_kernel, dim3(1u << kb), dim3(kBucketThreads), 0, st, ids, (int)R, (int)V, kb,
                           w.svals, w.skeys, w.rng, w.counts);
    } else {
        if (R > 0) {
            hipLaunchKernelGGL(emb_keys_kernel, dim3((unsigned)((R + 255) / 256)), dim3(256), 0, st, ids, R, V, w.keys,
                               w.vals);
            e = hipGetLastError();
            if (e != hipSuccess) return (int)e;
            size_t tb = w.temp_bytes;
            int end_bit = 1;
            while (end_bit < 32 && ((uint64_t)V >> end_bit) != 0) ++end_bit;   // keys are <= V
            e = sort_pairs(w.temp, tb, w.keys, w.skeys, w.vals, w.svals, R, end_bit, capturing(st), st);
            if (e != hipSuccess) return (int)e;
        }
        hipLaunchKernelGGL(emb_row_ranges_kernel, dim3((unsigned)((V + 255) / 256)), dim3(256), 0, st, w.skeys, R, V,
                           w.rng, w.counts);
    }
    e = hipGetLastError();
    if (e != hipSuccess) return (int)e;
    const int vec = (D % 8 == 0) && ((reinterpret_cast<uintptr_t>(grad) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
    int dev = 0;
    e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    size_t lds = 0;
    const int rc = z1detail::occupancy_lds(dev, kEmbWgPerCu, &lds);
    if (rc) return rc;
    // aten's kernel for few indices: its order, no heavy passes (nothing is listed for them)
    if (R < kSortMinRows) launch_rows<true>(D, V, lds, st, grad, w, padding_idx, scale, scale_mode, out);
    else launch_rows<false>(D, V, lds, st, grad, w, padding_idx, scale, scale_mode, out);
    e = hipGetLastError();
    if (e != hipSuccess) return (int)e;
    if (vec)
        hipLaunchKernelGGL(emb_heavy_parts_kernel<1>, dim3(kPartsGrid), dim3(kPartsThreads), 0, st, grad, D, w.svals,
                           w.skeys, w.rng, w.run_start, w.counts, scale, scale_mode, w.parts);
    else
        hipLaunchKernelGGL(emb_heavy_parts_kernel<0>, dim3(kPartsGrid), dim3(kPartsThreads), 0, st, grad, D, w.svals,
                           w.skeys, w.rng, w.run_start, w.counts, scale, scale_mode, w.parts);
    e = hipGetLastError();
    if (e != hipSuccess) return (int)e;
    hipLaunchKernelGGL(emb_heavy_chain_kernel, dim3(kChainGrid), dim3(kWave * kChainWaves), 0, st, w.parts, D,
                       w.rng, w.heavy_list, w.heavy_base, w.long_list, w.long_base, w.counts, scale, scale_mode,
                       out);
    e = hipGetLastError();
    return e == hipSuccess ? Z1_OK : (int)e;
}

}  // extern "C"
