// Token selection over device logit rows on gfx950: repetition penalty, greedy argmax and the
// sampled chain of sample_token (src/sampling.cpp:74-169), plus verify bookkeeping.
//
// select_slice_kernel covers all rows: grid (parts, rows), each 512-thread block owns an
// 8192-entry slice of one row, 16 values per thread held in registers. Per block: penalty on
// the slice's history ids (occurrence counts in LDS, each applied one occurrence at a time like
// the reference loop), then either the greedy rank maximum or {slice max, sum exp(l - slice max)
// in double, the slice's top-`want` ranks}. A row held by one slice finishes in the same
// block; otherwise select_merge_kernel (one block per row, second launch) merges the slices,
// ranks the global top-`want`, and runs top-p, top-k and the draw in reference order.
//
// The top-`want` of a block (block_top) is found by distance from the block's maximum: a
// 256-bin histogram of (max - v) locates the bin holding the want-th rank, every entry of a
// nearer bin is taken, and the boundary bin's entries are ranked exactly among themselves by
// the 64-bit (value desc, index asc) rank. Only the boundary bin needs exact work, and the
// histogram's atomics spread over 8 replicas. Blocks whose values do not bin usefully (all
// equal, non-finite extremes, an overfull boundary bin) fall back to a radix select on ranks.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>

#include "select_core.h"

namespace twd {


constexpr int kSliceThreads = 512;     // two slice blocks share a CU
constexpr int kSelPerThread = 16;
constexpr uint32_t kSlice = kSliceThreads * kSelPerThread;  // vocabulary entries per slice block
constexpr uint32_t kMaxParts = 64;    // vocab <= 64 * 8192 = 524288
constexpr int kMergeThreads = 256;
constexpr int kMergePerThread = kMaxParts * kMaxWant / kMergeThreads;  // 64

struct SelectArgs {
    uint32_t rows;
    uint32_t parts;
    uint32_t penalty_only;  // stop after the repetition penalty
    uint32_t one_pass;      // every row greedy: the slice blocks finish the rows themselves
    uint32_t epoch, next_epoch;
    twd_row_params p[TWD_MAX_ROWS + 1];  // verify samples up to K+1 rows
};

struct SelectBufs {
    float* logits;
    uint32_t vocab;
    uint64_t stride;
    const uint32_t* history;
    uint32_t* tokens;
    float* part_max;
    double* part_sum;
    uint32_t* part_flag;
    uint32_t* part_count;
    uint64_t* part_key;
    uint64_t* cand;
    uint64_t* gbest;  // one-pass greedy: per-row best ranks, zero between launches
    uint64_t* gctr;   // its arrival counter, kArriveWords words (grid_arrive)
};

// ... and per kernel: the slice kernel's penalty counts, then a copy of its values for the
// radix fallback, one entry per thread and slot so neither needs a barrier to hand over (two
// slice blocks fit on a CU); the merge kernel keeps every slice's ranks.
struct SliceShared {
    union {
        uint32_t cnt[kSlice];
        float vals[kSlice];
    } u;
    TopScratch t;
    SelCommon c;
};

struct MergeShared {
    uint64_t cand[kMaxParts * kMaxWant];  // every slice's ranks, packed
    uint32_t offs[kMaxParts + 1];         // where each slice's ranks start in cand
    TopScratch t;
    SelCommon c;
};

// After c.top[0..want) holds the row's shortlist and c.gmax/total/flag its statistics:
// the degenerate check of sampling.cpp:116-118, the shortlist sort, and steps 5-7.
__device__ __forceinline__ void finish_row(SelCommon& c, uint32_t want, const twd_row_params& p,
                           uint32_t* token_out, const float* row_logits, uint32_t vocab) {
    const int tid = threadIdx.x;
    if (c.flag != 0 || !(c.total > 0.0)) {
        if (tid == 0) *token_out = TWD_TOKEN_DEGENERATE;
        return;
    }
    block_sort_desc(c, want);
    const uint32_t tok = finish_sampled(c, want, p, c.total, RowSrc{row_logits, vocab, c.gmax, want});
    if (tid == 0) *token_out = tok;
}

// One-pass greedy finish (every row of the launch greedy, more than one slice): each slice block
// folds its best rank into its row's gbest slot with a returning atomic max and then counts
// itself in; the block that completes the count reads and clears every row's slot and writes
// the tokens. The protocol is the head's grid finish (device-scope atomics only, no fence):
// a returning atomic is performed at the memory-side coherence point before it returns, and
// the block waits for that return before it counts in, so every maximum precedes its
// block's arrival. The count is grid_arrive's (an epoch per launch, replay slots for captured
// launches).
__device__ __forceinline__ void select_greedy_finish(const SelectArgs& args, const SelectBufs& b, uint32_t row,
                                                     uint64_t k, SelCommon& c) {
    const int tid = threadIdx.x;
    if (tid == 0) {
        const unsigned long long seen = __hip_atomic_fetch_max(reinterpret_cast<unsigned long long*>(b.gbest + row),
                                                               static_cast<unsigned long long>(k), __ATOMIC_RELAXED,
                                                               __HIP_MEMORY_SCOPE_AGENT);
        c.red64[0] = seen;  // waits for the return: the maximum is performed before the count
        const uint32_t nb = gridDim.x * gridDim.y;
        const bool last = grid_arrive(reinterpret_cast<unsigned long long*>(b.gctr), nb, args.epoch, args.next_epoch);
        c.misc[7] = last ? 1u : 0u;
    }
    __syncthreads();
    if (!c.misc[7]) return;
    for (uint32_t r = tid; r < args.rows; r += blockDim.x) {
        const uint64_t kk = __hip_atomic_exchange(reinterpret_cast<unsigned long long*>(b.gbest + r), 0ull,
                                                  __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        b.tokens[r] = rank_index(kk);
    }
}

// SelectArgs is the first kernel argument, so it sits at offset 0 of the kernarg segment. The
// row's parameters are read through that pointer: indexing the by-value argument with
// blockIdx.y would make the compiler copy all of it into per-lane scratch memory.
__global__ __launch_bounds__(kSliceThreads) __attribute__((amdgpu_waves_per_eu(4)))
void select_slice_kernel(SelectArgs args_by_value, SelectBufs b) {
    constexpr int NT = kSliceThreads;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    SliceShared& sh = *reinterpret_cast<SliceShared*>(smem_raw);
#if __HIP_DEVICE_COMPILE__
    const SelectArgs& args =
        *reinterpret_cast<const SelectArgs*>(__builtin_amdgcn_kernarg_segment_ptr());
#else
    const SelectArgs& args = args_by_value;  // the host pass only parses kernel bodies
#endif
    const int tid = threadIdx.x;
    const uint32_t part = blockIdx.x, row = blockIdx.y;
    const uint32_t parts = args.parts;
    const twd_row_params p = args.p[row];
    float* lg = b.logits + static_cast<size_t>(row) * b.stride;
    const uint32_t lo = part * kSlice;
    const uint32_t hi = min(b.vocab, lo + kSlice);

    float v[kSelPerThread];
#pragma unroll
    for (int e = 0; e < kSelPerThread; ++e) {
        const uint32_t i = lo + tid + NT * e;
        v[e] = i < hi ? lg[i] : 0.0f;
    }
    for (uint32_t i = tid; i < kReps * kBins; i += NT) sh.t.hist[i] = 0;  // for block_top

    // ---- repetition penalty, sampling.cpp:74-90 ----
    if (p.repetition_penalty != 1.0f && p.history_len > 0) {
        // history ids in batches of kHistBatch per thread, each batch requested at once (one
        // round trip, not one per id); the first batch before the counts are cleared
        constexpr int kHistBatch = 8;
        const uint32_t* hist = b.history + p.history_offset;
        const uint32_t hlen = p.history_len;
        uint32_t ids[kHistBatch];
        auto fetch = [&](uint32_t j0) {
#pragma unroll
            for (int q = 0; q < kHistBatch; ++q) {
                const uint32_t j = j0 + tid + NT * q;
                ids[q] = j < hlen ? hist[j] : 0xFFFFFFFFu;  // never inside a slice
            }
        };
        auto count = [&]() {
#pragma unroll
            for (int q = 0; q < kHistBatch; ++q)
                if (ids[q] >= lo && ids[q] < hi) atomicAdd(&sh.u.cnt[ids[q] - lo], 1u);
        };
        fetch(0);
#pragma unroll
        for (int e = 0; e < kSelPerThread; ++e) sh.u.cnt[tid + NT * e] = 0;
        __syncthreads();
        count();
        for (uint32_t j0 = NT * kHistBatch; j0 < hlen; j0 += NT * kHistBatch) {
            fetch(j0);
            count();
        }
        __syncthreads();
        const float rp = p.repetition_penalty;
        const float limit = (p.softcap > 0.0f) ? p.softcap * 0.9999f : 0.0f;
#pragma unroll
        for (int e = 0; e < kSelPerThread; ++e) {
            const uint32_t n = sh.u.cnt[tid + NT * e];
            if (n == 0) continue;
            float x = v[e];
            for (uint32_t t = 0; t < n; ++t) {
                x = (x > 0.0f) ? (x / rp) : (x * rp);
                if (limit > 0.0f) {
                    const float lo_b = -limit;
                    x = (x < lo_b) ? lo_b : ((limit < x) ? limit : x);
                }
            }
            v[e] = x;
            lg[lo + tid + NT * e] = x;
        }
    }
    if (args.penalty_only) return;

    auto key_at = [&](int e) -> uint64_t {
        const uint32_t i = lo + tid + NT * e;
        return i < hi ? rank_key(v[e], i) : 0ull;
    };
    const bool greedy = p.temperature <= 0.0f;  // sampling.cpp:97: a NaN temperature samples
    if (greedy) {
        // ---- sampling.cpp:97-104 ----
        uint64_t k = 0;
#pragma unroll
        for (int e = 0; e < kSelPerThread; ++e) {
            const uint64_t r = key_at(e);
            k = r > k ? r : k;
        }
        k = block_max_u64<NT>(k, sh.c);
        if (parts == 1) {
            if (tid == 0) b.tokens[row] = rank_index(k);
            return;
        }
        if (args.one_pass) {
            select_greedy_finish(args, b, row, k, sh.c);
            return;
        }
        if (tid == 0) b.part_key[static_cast<size_t>(row) * parts + part] = k;
        return;
    }

    // a shortlist longer than kMaxWant: the long path finishes the row from its wave records
    if (p.top_k > static_cast<int32_t>(kMaxWant) && b.vocab > kMaxWant) return;
    // ---- sampled: slice statistics, sampling.cpp:109-118 ----
    // Any NaN makes the row degenerate, so the max only has to be right for NaN-free rows.
    uint32_t nan_seen = 0;
    float mx = -INFINITY, mn = INFINITY;
#pragma unroll
    for (int e = 0; e < kSelPerThread; ++e) {
        sh.u.vals[tid + NT * e] = v[e];  // the slot's count was read by this same thread
        if (lo + tid + NT * e < hi) {
            if (v[e] != v[e]) nan_seen = 1;
            mx = fmaxf(mx, v[e]);
            if (__builtin_isfinite(v[e])) mn = fminf(mn, v[e]);
        }
    }
    if (tid < 64) sh.c.exp2_tbl[tid] = kExp2Table[tid];
    block_stats<NT>(nan_seen, mx, mn, sh.c);  // its barriers also retire the penalty's counts
    const double dmx = static_cast<double>(mx);
    double s = 0.0;
#pragma unroll
    for (int e = 0; e < kSelPerThread; ++e)
        if (lo + tid + NT * e < hi) s += exp_for_sum(static_cast<double>(v[e]) - dmx, sh.c.exp2_tbl);
    s = block_sum_f64<NT>(s, sh.c);
    // A slice of -inf entries only adds exp(-inf - row max) = 0 to the row's sum whenever the
    // row has a finite maximum elsewhere (its own exp(-inf - -inf) would be NaN). If the whole
    // row is -inf every slice reports 0, the row total is 0 and the row is degenerate, as the
    // reference's NaN total makes it.
    if (mx == -INFINITY) s = 0.0;

    // ---- shortlist of this slice, sampling.cpp:120-137 ----
    const uint32_t want_row = (p.top_k > 0) ? min(static_cast<uint32_t>(p.top_k), b.vocab)
                                            : min(kMaxWant, b.vocab);
    const uint32_t n_here = hi - lo;
    const uint32_t want = min(want_row, n_here);
    auto val_at = [&](int e) -> float { return v[e]; };
    auto slow_val = [&](int e) -> float { return sh.u.vals[tid + NT * e]; };
    auto slow_key = [&](int e) -> uint64_t {
        const uint32_t i = lo + tid + NT * e;
        return i < hi ? rank_key(sh.u.vals[tid + NT * e], i) : 0ull;
    };
    uint64_t* out = (parts == 1) ? sh.c.top : b.cand + (static_cast<size_t>(row) * parts + part) * kMaxWant;
    block_top<NT, kSelPerThread>(val_at, key_at, slow_val, slow_key, kSelPerThread, mx, mn, want, out,
                                 sh.t, sh.c);

    if (parts > 1) {
        if (tid == 0) {
            const size_t o = static_cast<size_t>(row) * parts + part;
            b.part_max[o] = mx;
            b.part_sum[o] = s;
            b.part_flag[o] = nan_seen;
            b.part_count[o] = min(sh.c.misc[4], want);  // fewer only when NaNs hold no rank
        }
        return;  // select_merge_kernel finishes the row
    }
    if (tid == 0) {
        sh.c.gmax = mx;
        sh.c.total = s;
        sh.c.flag = nan_seen;
    }
    __syncthreads();
    finish_row(sh.c, want_row, p, b.tokens + row, b.logits + static_cast<size_t>(row) * b.stride, b.vocab);
}

// Second launch when a row spans several slices: global max, the rescaled sum of exponentials,
// the global shortlist from every slice's candidates, then the draw. One block per row.
__global__ __launch_bounds__(kMergeThreads) void select_merge_kernel(SelectArgs args_by_value, SelectBufs b) {
    constexpr int NT = kMergeThreads;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    MergeShared& sh = *reinterpret_cast<MergeShared*>(smem_raw);
#if __HIP_DEVICE_COMPILE__
    const SelectArgs& args =
        *reinterpret_cast<const SelectArgs*>(__builtin_amdgcn_kernarg_segment_ptr());
#else
    const SelectArgs& args = args_by_value;
#endif
    const int tid = threadIdx.x, lane = tid & 63;
    const uint32_t row = blockIdx.x;
    const uint32_t parts = args.parts;  // <= kMaxParts = 64: one lane of wave 0 per slice
    const twd_row_params p = args.p[row];
    const size_t o = static_cast<size_t>(row) * parts;

    if (p.temperature <= 0.0f) {  // greedy: the best rank over the slices
        if (tid < 64) {
            const uint64_t m = wave_max_u64(static_cast<uint32_t>(lane) < parts ? b.part_key[o + lane] : 0ull);
            if (tid == 0) b.tokens[row] = rank_index(m);
        }
        return;
    }
    const uint32_t want_row = (p.top_k > 0) ? min(static_cast<uint32_t>(p.top_k), b.vocab)
                                            : min(kMaxWant, b.vocab);
    if (want_row > kMaxWant) return;  // the long path finishes the row
    for (uint32_t i = tid; i < kReps * kBins; i += NT) sh.t.hist[i] = 0;  // for block_top
    // Wave 0: global max and NaN flag over the slices, the row sum
    // sum_q part_sum[q] * exp(part_max[q] - max), and where each slice's ranks go.
    if (tid < 64) {
        const bool live = static_cast<uint32_t>(lane) < parts;
        const float pm = live ? b.part_max[o + lane] : -INFINITY;
        const double ps = live ? b.part_sum[o + lane] : 0.0;
        uint32_t fl = live ? b.part_flag[o + lane] : 0u;
        const uint32_t cnt = live ? b.part_count[o + lane] : 0u;
        float gm = pm;
        uint32_t x = cnt;  // inclusive prefix sum of the counts
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) {
            gm = fmaxf(gm, __shfl_xor(gm, m));
            fl |= __shfl_xor(fl, m);
        }
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t y = __shfl_up(x, off);
            if (lane >= off) x += y;
        }
        double contrib = live ? ps * exp(static_cast<double>(pm) - static_cast<double>(gm)) : 0.0;
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) contrib += __shfl_xor(contrib, m);
        sh.offs[lane] = x - cnt;
        if (lane == 63) sh.offs[kMaxParts] = x;
        if (lane == 0) {
            sh.c.gmax = gm;
            sh.c.total = contrib;
            sh.c.flag = fl;
        }
    }
    __syncthreads();
    const uint32_t n_cand = sh.offs[kMaxParts];
    const float gm = sh.c.gmax;
    // every slice's ranks, packed into cand[0 .. n_cand)
    float cmn = INFINITY;
    const uint32_t nf = parts * want_row;
    constexpr int kGatherBatch = 4;  // loads requested together, then stored
    for (uint32_t f0 = 0; f0 < nf; f0 += NT * kGatherBatch) {
        uint64_t kk[kGatherBatch];
        uint32_t at[kGatherBatch];
#pragma unroll
        for (int u = 0; u < kGatherBatch; ++u) {
            const uint32_t f = f0 + tid + NT * u;
            at[u] = 0xFFFFFFFFu;
            kk[u] = 0;
            if (f < nf) {
                const uint32_t q = f / want_row, slot = f % want_row;
                const uint32_t a = sh.offs[q] + slot;
                if (a < sh.offs[q + 1]) {
                    at[u] = a;
                    kk[u] = b.cand[(o + q) * kMaxWant + slot];
                }
            }
        }
#pragma unroll
        for (int u = 0; u < kGatherBatch; ++u) {
            if (at[u] == 0xFFFFFFFFu) continue;
            sh.cand[at[u]] = kk[u];
            const float x = rank_value(kk[u]);
            if (kk[u] != 0 && __builtin_isfinite(x)) cmn = fminf(cmn, x);
        }
    }
    uint32_t no_flag = 0;
    float no_max = -INFINITY;
    block_stats<NT>(no_flag, no_max, cmn, sh.c);  // its barriers also publish sh.cand
    auto merge_key = [&](int e) -> uint64_t {
        const uint32_t f = tid + NT * e;
        return f < n_cand ? sh.cand[f] : 0ull;
    };
    auto merge_val = [&](int e) -> float { return rank_value(merge_key(e)); };
    const int per = static_cast<int>((n_cand + NT - 1) / NT);
    block_top<NT, kMergePerThread>(merge_val, merge_key, merge_val, merge_key, per, gm, cmn, want_row,
                                   sh.c.top, sh.t, sh.c);
    finish_row(sh.c, want_row, p, b.tokens + row, b.logits + static_cast<size_t>(row) * b.stride, b.vocab);
}

// ---- after the head's sample mode (or the wave-record pass): one block per row --------------------
// sample_merge_row (select_core.h) finishes each row from its per-64-entry records.
template <uint32_t RSH, uint32_t PER>
__global__ __launch_bounds__(kSmThreads) void select_sample_merge_kernel(SelectArgs args_by_value,
                                                                         SampleMergeBufs b) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    SampleMergeShared& sh = *reinterpret_cast<SampleMergeShared*>(smem_raw);
#if __HIP_DEVICE_COMPILE__
    const SelectArgs& args =
        *reinterpret_cast<const SelectArgs*>(__builtin_amdgcn_kernarg_segment_ptr());
#else
    const SelectArgs& args = args_by_value;
#endif
    const uint32_t row = blockIdx.x;
    sample_merge_row_per<PER, RSH>(args.p[row], row, b, sh);
}

// The merge by its record size and by the records per thread that its rows need, one kernel for each:
// the launch is one block a row, bound by the chain of its phases and the instructions of its 16 waves
// on one CU, so a thread that holds one record should not step through four (binning, exponential and
// candidate test each, at every q). One kernel with a branch between the counts is no substitute: with
// all of them in it the same rows took 0.5 to 1.5 us more. The record pass and this kernel, top_k 40,
// one row, before (4 or 8 a thread) and after: V = 32,003 11.8 and 10.7 us, V = 100,003 10.6 and 9.9,
// V = 262,144 (4 a thread either way) 11.5 and 11.2; 8 rows 12.2 and 11.1, 13.2 and 12.4, 13.6 and 13.5.
using MergeKernel = void (*)(SelectArgs, SampleMergeBufs);
// Records of 16 entries are at most 4,096 (one tile per wave), records of 32 from 2,049 to 4,096 (two):
// counts outside those are no call's (null).
template <uint32_t RSH>
MergeKernel merge_kernel(uint32_t waves) {
    if constexpr (RSH != 5) {
        if (waves <= kSmThreads) return select_sample_merge_kernel<RSH, 1>;
        if (waves <= kSmThreads * 2) return select_sample_merge_kernel<RSH, 2>;
    }
    if (waves <= kSmThreads * (kSmPer / 2)) return select_sample_merge_kernel<RSH, kSmPer / 2>;
    if constexpr (RSH == 6) return select_sample_merge_kernel<RSH, kSmPer>;
    return nullptr;
}

// ---- shortlists longer than 256: top_k > 256 -------------------------------------------------------
//
// sample_token takes any top_k: its shortlist is the top want = min(top_k, V) entries in the
// order (value desc, index asc), and steps 5-7 run over all of them (sampling.cpp:120-168).
// Rows with temperature > 0 and want > 256 are finished from the penalised logits and the same
// wave records as the shorter rows (so the same row max and total): those of up to kWideMax entries
// by the wide kernels below, longer ones by these:
//   * long_gather_kernel, one block per row: records_stats, then every entry of a candidate wave
//     (maximum in a bin <= b*) that lies in a bin <= b*, into the row's sort buffer in any
//     order. Every top-`want` entry is among them. The buffer is padded with zero ranks (below
//     every real rank) to a power of two, its sort length;
//   * a bitonic sort of each buffer into descending order: long_sort_tile_kernel sorts tiles of
//     kSortTile ranks in LDS (alternating directions); each longer stage k runs its cross-tile
//     steps (long_sort_step_kernel, one launch per step) and then its in-tile steps
//     (long_sort_merge_kernel). The launches cover the longest possible buffer; a block past its
//     row's sort length, or of a stage longer than it, returns at once;
//   * long_finish_kernel, one block per row: steps 5-7 over the sorted ranks, kFinTile at a
//     time. The block forms the terms exp(l - max) / total and exp((l - max) / T) in LDS with the
//     reference's expressions; the two running sums then go in reference order on two lanes of
//     wave 0 (finish_sampled's loop), and the running sums of the temperature weights are kept in
//     memory. After the cut (top-p, then top-k), r = u * denom and the draw is the first running
//     sum >= r: the running sums never decrease, so a search over the tiles' last sums, then
//     over one tile, finds it.
constexpr int kLongThreads = 1024;
constexpr uint32_t kSortTile = 8192;  // ranks sorted in LDS by one block (64 KB)
constexpr int kStepThreads = 256;
constexpr uint32_t kFinTile = 2048;   // shortlist entries per tile of the finish

struct LongArgs {
    uint32_t n;                          // long rows in the launch
    uint32_t row[TWD_MAX_ROWS + 1];      // each one's row in the call
    twd_row_params p[TWD_MAX_ROWS + 1];  // and its parameters
};

struct LongBufs {
    const float* logits;  // [rows][stride], penalised
    uint64_t stride;
    uint32_t vocab;
    uint32_t waves;       // records per row
    uint32_t rec_shift;   // log2 of the entries per record
    SampleStats st;       // [row][waves]
    uint64_t npad;        // sort buffer per long row: a power of two >= vocab
    uint64_t* keys;       // [n][npad]
    double* pre;          // [n][npad] running sums of the temperature weights
    uint32_t* len;        // [n] sort length (0: the row is already finished)
    float* gmax;          // [n]
    double* total;        // [n]
    struct WideState* wide;  // [n] rows of up to kWideMax entries
    uint32_t* tokens;
};

struct LongGatherShared {
    uint32_t cwave[kSampleMaxWaves];
    TopScratch t;
    SelCommon c;
};

// The long-path kernels read LongArgs (the first kernel argument) through the kernarg segment
// pointer: indexing the by-value argument with blockIdx would copy it to scratch memory.
#if __HIP_DEVICE_COMPILE__
#define TWD_LONG_ARGS(byval) \
    (*reinterpret_cast<const LongArgs*>(__builtin_amdgcn_kernarg_segment_ptr()))
#else
#define TWD_LONG_ARGS(byval) (byval)
#endif

__global__ __launch_bounds__(kLongThreads) void long_gather_kernel(LongArgs args_by_value, LongBufs b) {
    constexpr int NT = kLongThreads;
    static_assert(NT == kSmThreads, "records_stats' block");
    extern __shared__ __align__(16) unsigned char smem_raw[];
    LongGatherShared& sh = *reinterpret_cast<LongGatherShared*>(smem_raw);
    const LongArgs& args = TWD_LONG_ARGS(args_by_value);
    const int tid = threadIdx.x, lane = tid & 63;
    const uint32_t j = blockIdx.x;
    const uint32_t row = args.row[j];
    const twd_row_params p = args.p[j];
    const uint32_t W = b.waves;
    const size_t o = static_cast<size_t>(row) * W;
    const float* lg = b.logits + static_cast<size_t>(row) * b.stride;
    uint64_t* keys = b.keys + static_cast<size_t>(j) * b.npad;

    if (tid < 64) sh.c.exp2_tbl[tid] = kExp2Table[tid];
    uint64_t key[kSmPer];
    double wsum[kSmPer];
#pragma unroll
    for (uint32_t q = 0; q < kSmPer; ++q) {
        const uint32_t i = tid + NT * q;
        key[q] = i < W ? b.st.key[o + i] : 0ull;
        wsum[q] = i < W ? b.st.sum[o + i] : 0.0;
    }
    for (uint32_t i = tid; i < kReps * kBins; i += NT) sh.t.hist[i] = 0;
    const uint32_t want = min(static_cast<uint32_t>(p.top_k), b.vocab);
    float wm[kSmPer];
    bool live[kSmPer];
    uint32_t nan = 0;
#pragma unroll
    for (uint32_t q = 0; q < kSmPer; ++q) {
        live[q] = key[q] != 0;
        wm[q] = live[q] ? rank_value(key[q]) : -INFINITY;
        nan |= wsum[q] != wsum[q] ? 1u : 0u;
    }
    const RecStats rs = records_stats(live, wm, nan, wsum, fixed_ref(b.st.cap, p), want, sh.t, sh.c);
    if (rs.degenerate) {  // sampling.cpp:116-118
        if (tid == 0) {
            b.tokens[row] = TWD_TOKEN_DEGENERATE;
            b.len[j] = 0;
        }
        return;
    }
    // the candidate waves, in any order (at most W <= kSampleMaxWaves)
#pragma unroll
    for (uint32_t q = 0; q < kSmPer; ++q) {
        const uint32_t i = tid + NT * q;
        const bool is_cand = key[q] != 0 && rec_bin(rs, wm[q]) <= rs.bstar;
        const uint64_t mask = __ballot(is_cand);
        if (mask != 0) {
            const int leader = __ffsll(static_cast<long long>(mask)) - 1;
            uint32_t base = 0;
            if (lane == leader) base = atomicAdd(&sh.c.misc[3], static_cast<uint32_t>(__popcll(mask)));
            base = __builtin_amdgcn_readlane(base, leader);
            if (is_cand) {
                const uint32_t below = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(mask >> 32),
                                                                  __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(mask), 0u));
                sh.cwave[base + below] = i;
            }
        }
    }
    __syncthreads();
    const uint32_t rsh = b.rec_shift, rmask = (1u << rsh) - 1u;
    const uint32_t nent = sh.c.misc[3] << rsh;
    // the survivors into the sort buffer, eight loads requested at a time
    constexpr uint32_t kBatch = 8;
    const uint32_t per = (nent + NT - 1) / NT;
    for (uint32_t i0 = 0; i0 < per; i0 += kBatch) {
        float v[kBatch];
        uint32_t r[kBatch];
#pragma unroll
        for (uint32_t q = 0; q < kBatch; ++q) {
            const uint32_t f = (i0 + q) * NT + static_cast<uint32_t>(tid);
            r[q] = 0xFFFFFFFFu;
            v[q] = 0.0f;
            if (i0 + q < per && f < nent) {
                const uint32_t rr = (sh.cwave[f >> rsh] << rsh) + (f & rmask);
                if (rr < b.vocab) {
                    r[q] = rr;
                    v[q] = lg[rr];
                }
            }
        }
#pragma unroll
        for (uint32_t q = 0; q < kBatch; ++q) {
            const bool keep = r[q] != 0xFFFFFFFFu && rec_bin(rs, v[q]) <= rs.bstar;
            wave_put(keep, keep ? rank_key(v[q], r[q]) : 0ull, &sh.c.misc[4], keys, static_cast<uint32_t>(b.npad));
        }
    }
    __syncthreads();
    const uint32_t n = sh.c.misc[4];
    uint32_t len = 1;
    while (len < n) len <<= 1;
    for (uint32_t i = n + tid; i < len; i += NT) keys[i] = 0ull;
    if (tid == 0) {
        b.len[j] = len;
        b.gmax[j] = rs.gm;
        b.total[j] = rs.total;
    }
}

// One compare-exchange of the bitonic network over a row's buffer (global positions): the pair
// (i, i | jj) in stage k is put in descending order when bit k of i is clear, ascending when it
// is set, so the last stage (k = length) leaves the whole buffer descending.
__device__ __forceinline__ void bitonic_pair(uint64_t& a, uint64_t& c, uint64_t gi, uint64_t k) {
    const bool desc = (gi & k) == 0;
    if (desc ? a < c : a > c) {
        const uint64_t t = a;
        a = c;
        c = t;
    }
}

// steps jj = j0, j0 / 2, .., 1 of stage k on the LDS tile s of `t` ranks starting at global base
__device__ __forceinline__ void bitonic_tile_steps(uint64_t* s, uint32_t t, uint64_t base, uint64_t k, uint32_t j0) {
    for (uint32_t jj = j0; jj > 0; jj >>= 1) {
        for (uint32_t q = threadIdx.x; q < t / 2; q += blockDim.x) {
            const uint32_t i = ((q & ~(jj - 1)) << 1) | (q & (jj - 1));
            uint64_t a = s[i], c = s[i | jj];
            bitonic_pair(a, c, base + i, k);
            s[i] = a;
            s[i | jj] = c;
        }
        __syncthreads();
    }
}

__global__ __launch_bounds__(kLongThreads) void long_sort_tile_kernel(LongBufs b, uint32_t tile) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    uint64_t* s = reinterpret_cast<uint64_t*>(smem_raw);
    const uint32_t j = blockIdx.y;
    const uint32_t len = b.len[j];
    const uint64_t base = static_cast<uint64_t>(blockIdx.x) * tile;
    if (base >= len) return;  // the whole block
    const uint32_t t = min(tile, len);  // both powers of two
    uint64_t* keys = b.keys + static_cast<size_t>(j) * b.npad + base;
    for (uint32_t i = threadIdx.x; i < t; i += blockDim.x) s[i] = keys[i];
    __syncthreads();
    for (uint32_t k = 2; k <= t; k <<= 1) bitonic_tile_steps(s, t, base, k, k >> 1);
    for (uint32_t i = threadIdx.x; i < t; i += blockDim.x) keys[i] = s[i];
}

__global__ __launch_bounds__(kStepThreads) void long_sort_step_kernel(LongBufs b, uint32_t k, uint32_t jj) {
    const uint32_t j = blockIdx.y;
    const uint32_t len = b.len[j];
    const uint64_t q = static_cast<uint64_t>(blockIdx.x) * kStepThreads + threadIdx.x;
    if (k > len || 2 * q >= len) return;
    const uint64_t i = ((q & ~static_cast<uint64_t>(jj - 1)) << 1) | (q & (jj - 1));
    uint64_t* keys = b.keys + static_cast<size_t>(j) * b.npad;
    uint64_t a = keys[i], c = keys[i | jj];
    bitonic_pair(a, c, i, k);
    keys[i] = a;
    keys[i | jj] = c;
}

__global__ __launch_bounds__(kLongThreads) void long_sort_merge_kernel(LongBufs b, uint32_t tile, uint32_t k) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    uint64_t* s = reinterpret_cast<uint64_t*>(smem_raw);
    const uint32_t j = blockIdx.y;
    const uint32_t len = b.len[j];
    const uint64_t base = static_cast<uint64_t>(blockIdx.x) * tile;
    if (k > len || base >= len) return;  // the whole block; here len >= k > tile
    uint64_t* keys = b.keys + static_cast<size_t>(j) * b.npad + base;
    for (uint32_t i = threadIdx.x; i < tile; i += blockDim.x) s[i] = keys[i];
    __syncthreads();
    bitonic_tile_steps(s, tile, base, k, tile >> 1);
    for (uint32_t i = threadIdx.x; i < tile; i += blockDim.x) keys[i] = s[i];
}

struct LongFinishShared {
    double e[kFinTile];  // exp(l - max) / total, then lane 1's running sums
    double q[kFinTile];  // exp((l - max) / T), then lane 0's running sums
    double base;         // lane 1's running sum before the tile
    double total;        // the reference's row total, when the cut takes it
    uint32_t misc[4];
    uint32_t best;
};

// Steps 5-7 of long row j over its sorted ranks in b.keys. One block of kLongThreads threads; every
// thread calls. Inlined into its kernel: as a function called with these references it reads the
// arguments and the LDS through generic pointers, 25 to 65 us a row (V = 262,144, top_k = 5,000:
// 508 and 574 us).
__device__ __forceinline__ void long_finish_row(const LongArgs& args, const LongBufs& b, uint32_t j, float gmax,
                                             double total, LongFinishShared& sh) {
    constexpr int NT = kLongThreads;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t row = args.row[j];
    const twd_row_params p = args.p[j];
    const uint64_t* keys = b.keys + static_cast<size_t>(j) * b.npad;
    double* pre = b.pre + static_cast<size_t>(j) * b.npad;
    const uint32_t want = min(static_cast<uint32_t>(p.top_k), b.vocab);
    const double mx = static_cast<double>(gmax);
    const double td = static_cast<double>(p.temperature);
    const bool topp = p.top_p < 1.0f;
    const double pp = static_cast<double>(p.top_p);
    constexpr uint32_t kChunk = 16;
    uint32_t cut = want;
    // a second pass with the reference's own row total when the first pass's cut lies within
    // total_tol of p (see finish_sums_exact)
    for (int pass = 0;; ++pass) {
        double run = 0.0;  // wave 0: lane 0's sum of the weights, lane 1's top-p sum
        uint32_t tl = 0;   // the last tile's first entry
        cut = want;
        if (tid == 0) sh.misc[0] = 0;
        for (uint32_t t0 = 0; t0 < want; t0 += kFinTile) {
            tl = t0;
            const uint32_t cnt = min(kFinTile, want - t0);
            // steps 5 and 7's terms, as sampling.cpp:145 and :157 form them
            for (uint32_t i = tid; i < cnt; i += NT) {
                const double l = static_cast<double>(rank_value(keys[t0 + i]));
                sh.q[i] = exp_libm((l - mx) / td);
                if (topp) sh.e[i] = exp_libm(l - mx) / total;
            }
            __syncthreads();
            if (wave == 0 && lane < 2) {
                // lane 0 reads q and stores its running sums over q; lane 1 does the same over e
                // (over q when top-p is off: its sums are then never used)
                double* src = (lane == 0 || !topp) ? sh.q : sh.e;
                if (lane == 1) sh.base = run;  // the top-p sum before the tile
                double x[kChunk];
#pragma unroll
                for (uint32_t jj = 0; jj < kChunk; ++jj) x[jj] = src[min(jj, cnt - 1)];
                for (uint32_t i0 = 0; i0 < cnt; i0 += kChunk) {
                    double xn[kChunk], pr[kChunk];
                    if (i0 + kChunk < cnt) {
#pragma unroll
                        for (uint32_t jj = 0; jj < kChunk; ++jj) xn[jj] = src[min(i0 + kChunk + jj, cnt - 1)];
                    }
#pragma unroll
                    for (uint32_t jj = 0; jj < kChunk; ++jj) {
                        run += x[jj];
                        pr[jj] = run;
                    }
                    uint32_t hit = 0;
#pragma unroll
                    for (uint32_t jj = 0; jj < kChunk; ++jj) {
                        src[i0 + jj] = pr[jj];  // i0 + jj < cnt rounded up to kChunk <= kFinTile
                        hit |= (pr[jj] >= pp ? 1u : 0u) << jj;
                    }
                    uint32_t h1 = __builtin_amdgcn_readlane(hit, 1);
                    h1 &= cnt - i0 >= kChunk ? 0xFFFFu : ((1u << (cnt - i0)) - 1u);
                    if (topp && h1 != 0) {  // lane 0's sums cover the cut
                        if (lane == 0) sh.misc[0] = t0 + i0 + static_cast<uint32_t>(__builtin_ctz(h1)) + 1;
                        break;
                    }
#pragma unroll
                    for (uint32_t jj = 0; jj < kChunk; ++jj) x[jj] = xn[jj];
                }
            }
            __syncthreads();
            const uint32_t c = sh.misc[0];  // the cut, once the top-p sum has reached p
            const uint32_t keep = c != 0 ? c - t0 : cnt;
            for (uint32_t i = tid; i < keep; i += NT) pre[t0 + i] = sh.q[i];
            if (c != 0) {
                cut = c;
                break;
            }
            __syncthreads();  // the next tile's terms overwrite sh
        }
        if (!topp || pass > 0) break;
        // the last tile's top-p sums are in sh.e: the one at the cut (when it reached p) and the
        // one before it decide (as in finish_sums_exact)
        if (tid == 0) {
            const double tc = total_tol(b.vocab);
            const double hi = sh.e[cut - 1 - tl];
            const double lo = cut >= 2 ? (cut - 2 >= tl ? sh.e[cut - 2 - tl] : sh.base) : 0.0;
            const bool near = (hi >= pp && hi <= pp * (1.0 + tc)) ||
                              (cut >= 2 && lo >= pp * (1.0 - tc) && lo <= pp * (1.0 + tc));
            sh.misc[2] = near ? 1u : 0u;
        }
        __syncthreads();
        if (sh.misc[2] == 0) break;
        if (wave == 0) {
            const double t = exact_row_total(RowSrc{b.logits + static_cast<size_t>(row) * b.stride, b.vocab,
                                                    gmax, 0u}, sh.e);
            if (lane == 0) sh.total = t;
        }
        __syncthreads();
        total = sh.total;
    }
    if (p.top_k > 0 && cut > static_cast<uint32_t>(p.top_k)) cut = static_cast<uint32_t>(p.top_k);
    if (cut < 1) cut = 1;
    if (tid == 0) sh.best = cut - 1;  // the reference's fallback: the last survivor
    __syncthreads();                  // also publishes pre (block scope)
    const double r = static_cast<double>(p.uniform) * pre[cut - 1];  // r = u * denom
    // the first tile whose last running sum (within the cut) reaches r, then its first entry
    const uint32_t ntiles = (cut + kFinTile - 1) / kFinTile;
    if (tid == 0) sh.misc[1] = ntiles - 1;
    __syncthreads();
    for (uint32_t t = tid; t < ntiles; t += NT)
        if (pre[min((t + 1) * kFinTile, cut) - 1] >= r) atomicMin(&sh.misc[1], t);
    __syncthreads();
    const uint32_t t0 = sh.misc[1] * kFinTile, t1 = min(t0 + kFinTile, cut);
    for (uint32_t i = t0 + tid; i < t1; i += NT)
        if (pre[i] >= r) atomicMin(&sh.best, i);
    __syncthreads();
    if (tid == 0) b.tokens[row] = rank_index(keys[sh.best]);
}

__global__ __launch_bounds__(kLongThreads) void long_finish_kernel(LongArgs args_by_value, LongBufs b) {
    __shared__ LongFinishShared sh;
    const LongArgs& args = TWD_LONG_ARGS(args_by_value);
    const uint32_t j = blockIdx.x;
    if (b.len[j] == 0) return;  // degenerate: long_gather_kernel wrote its token
    long_finish_row(args, b, j, b.gmax[j], b.total[j], sh);
}

// long_finish_row where it is seldom reached: a call, so that the kernel around it keeps its registers.
__device__ __noinline__ void long_finish_row_call(const LongArgs& args, const LongBufs& b, uint32_t j, float gmax,
                                                  double total, LongFinishShared& sh) {
    long_finish_row(args, b, j, gmax, total, sh);
}

// ---- shortlists of 257 to kWideMax entries ---------------------------------------------------------
//
// The long path above moves every candidate through memory and sorts it over as many launches as the
// longest possible buffer needs: 25 launches and 150 us for eight rows of V = 262,144 at
// top_k = 1,000, most of them sort stages that no row reached. A shortlist of up to kWideMax
// entries fits a CU's LDS, with room for the entries that share its last bin:
//   * wide_filter_kernel<false>, `parts` blocks per row: the row's statistics and b* from its
//     records, as the merge takes them, then the entries in bins <= b* of the block's share of the
//     candidate records (every parts-th one), appended to the row's list in memory. One block per
//     row is not enough for this: some 50 instructions per entry, 25 us for 65,000 entries on one CU;
//   * where the records are too few to bound the shortlist (want near or past their number: every
//     entry would be a candidate), wide_filter_kernel<true> first counts the entries in kFineBins
//     bins of distance from the row max, and the list takes the fine bins up to the one that holds
//     the want-th entry;
//   * wide_finish_kernel, one block per row, all in LDS: a bucket sort (an entry's place is its fine
//     bin's start plus the entries of the bin above it; a bitonic sort when a bin holds more than
//     kWideBucket), then steps 5-7 by prefix sums over the block with finish_sums_par's margins. Its
//     bound holds here: a running sum of up to 4,096 terms lies within 4,096 x 2^-53 of the exact
//     one, so the parallel prefixes and the reference's differ by less than 2^-40, against the
//     margin of 2^-36. A decision within the margin takes long_finish_row's sums, the reference's
//     own. A list longer than kWideCap (ties) is gathered again by this block, by fine bins and, if
//     the last bin alone is too long, above the want-th rank that a radix select finds.
// Entries that dead_distance marks can be neither cut nor drawn and are left out, as in the merge.
// Eight rows of V = 262,144 at top_k = 1,000: 150 -> 28.4 us.
constexpr uint32_t kWideMax = 4096;    // longest shortlist
constexpr uint32_t kWideCap = 8192;    // longest list
constexpr uint32_t kFineBins = 2048;
constexpr uint32_t kWideBucket = 192;  // entries of one fine bin ranked against each other
constexpr uint32_t kWideLast = 64;     // entries of the last one that are
constexpr uint32_t kPartCap = 4096;    // list entries of one filter block

// The records bound the shortlist: with want below three quarters of their number, the entries above
// the want-th maximum are some 1.4 times as many (64 entries per record, in any order).
__device__ __host__ inline bool wide_needs_bins(uint32_t want, uint32_t waves) {
    return 4u * want > 3u * (waves < 4096u ? waves : 4096u);
}

// A draw outside [0, 1) can fall past every weight, on the last survivor, dead or not.
__device__ __forceinline__ double wide_dead(const twd_row_params& p) {
    return p.uniform >= 0.0f && p.uniform < 1.0f ? dead_distance(p) : -INFINITY;
}

struct FineBin {
    float gm, scale;
    __device__ __forceinline__ uint32_t operator()(float x) const {
        const float dist = (gm - x) * scale;  // scale 0: no bins
        return dist < static_cast<float>(kFineBins - 1) ? static_cast<uint32_t>(dist) : kFineBins - 1;
    }
};

// The records' bins in eight parts each; over twice their range where the shortlist can reach below
// the smallest record maximum, which is where that range ends.
__device__ __forceinline__ FineBin fine_bins(float gm, float scale, bool beyond) {
    return FineBin{gm, scale * (static_cast<float>(kFineBins) / kBins) * (beyond ? 0.5f : 1.0f)};
}

// hist[0..kFineBins) to its inclusive prefix sums: two bins per thread.
__device__ __forceinline__ void fine_scan(uint32_t* hist, uint32_t* wsum) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    static_assert(kFineBins == 2 * kLongThreads, "two bins per thread");
    const uint32_t a = hist[2 * tid], b = hist[2 * tid + 1];
    uint32_t x = wave_incl_scan_u32(a + b);
    if (lane == 63) wsum[wave] = x;
    __syncthreads();
    for (int w = 0; w < wave; ++w) x += wsum[w];
    hist[2 * tid] = x - b;
    hist[2 * tid + 1] = x;
    __syncthreads();
}

// The first fine bin by which `want` entries have been counted (the last one when fewer are there):
// hist holds inclusive sums. Every thread calls; *out is shared.
__device__ __forceinline__ uint32_t fine_bound(const uint32_t* hist, uint32_t want, uint32_t* out) {
    if (threadIdx.x == 0) *out = kFineBins - 1;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < kFineBins; i += blockDim.x)
        if (hist[i] >= want && (i == 0 || hist[i - 1] < want)) *out = i;  // one writer at most
    __syncthreads();
    return *out;
}

// f(value, row, in range) over the entries of the records listed in cwave[0..ncw), kBatch loads per
// thread requested together; the same trip count in every thread.
template <typename F>
__device__ __forceinline__ void for_entries(const uint16_t* cwave, uint32_t ncw, uint32_t rsh, uint32_t vocab,
                                            const float* lg, F&& f) {
    constexpr int NT = kLongThreads;
    constexpr uint32_t kBatch = 8;
    const uint32_t rmask = (1u << rsh) - 1u, nent = ncw << rsh, per = (nent + NT - 1) / NT;
    for (uint32_t i0 = 0; i0 < per; i0 += kBatch) {
        float v[kBatch];
        uint32_t r[kBatch];
        bool in[kBatch];
#pragma unroll
        for (uint32_t q = 0; q < kBatch; ++q) {
            const uint32_t e = (i0 + q) * NT + threadIdx.x;
            r[q] = e < nent ? (static_cast<uint32_t>(cwave[e >> rsh]) << rsh) + (e & rmask) : 0xFFFFFFFFu;
            in[q] = r[q] < vocab;
        }
#pragma unroll
        for (uint32_t q = 0; q < kBatch; ++q) v[q] = lg[in[q] ? r[q] : 0u];
        f(v, r, in);
    }
}

// A row's statistics from the filter's first block for the finish, its list's length and its fine
// counts. n and hist are zero between calls: the finish clears them.
struct WideState {
    double total;
    float gm, scale;
    uint32_t bstar, degenerate;
    uint32_t n;
    uint32_t hist[kFineBins];
};

struct WideFilterShared {
    uint64_t keys[kPartCap];
    uint16_t cwave[kSampleMaxWaves];
    uint32_t hist[kFineBins];
    uint32_t wsum[16], base, bound;
    TopScratch t;
    SelCommon c;
};

template <bool COUNT>
__global__ __launch_bounds__(kLongThreads) void wide_filter_kernel(LongArgs args_by_value, LongBufs b) {
    constexpr int NT = kLongThreads;
    static_assert(NT == kSmThreads, "records_stats' block");
    extern __shared__ __align__(16) unsigned char smem_raw[];
    WideFilterShared& sh = *reinterpret_cast<WideFilterShared*>(smem_raw);
    const LongArgs& args = TWD_LONG_ARGS(args_by_value);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t part = blockIdx.x, parts = gridDim.x, j = blockIdx.y;
    const uint32_t row = args.row[j];
    const twd_row_params p = args.p[j];
    const uint32_t W = b.waves;
    const size_t o = static_cast<size_t>(row) * W;
    const float* lg = b.logits + static_cast<size_t>(row) * b.stride;
    WideState& st = b.wide[j];
    const uint32_t want = min(static_cast<uint32_t>(p.top_k), b.vocab);  // <= kWideMax
    const bool binned = wide_needs_bins(want, W);
    if (COUNT && !binned) return;
    const double dead = wide_dead(p);

    float wm[kSmPer];
    bool live[kSmPer];
    uint32_t nan = 0;
#pragma unroll
    for (uint32_t q = 0; q < kSmPer; ++q) {
        const uint32_t i = tid + NT * q;
        live[q] = i < W;
        wm[q] = live[q] ? b.st.max[o + i] : -INFINITY;
        nan |= wm[q] != wm[q] ? 1u : 0u;
    }
    float gm, scale;
    uint32_t bstar = 0;
    if (COUNT || !binned) {
        // the statistics; the first block also the row total
        double wsum[kSmPer];
        if (tid < 64) sh.c.exp2_tbl[tid] = kExp2Table[tid];
        if (part == 0) {
#pragma unroll
            for (uint32_t q = 0; q < kSmPer; ++q) wsum[q] = live[q] ? b.st.sum[o + tid + NT * q] : 0.0;
        }
        for (uint32_t i = tid; i < kReps * kBins; i += NT) sh.t.hist[i] = 0;
        if constexpr (COUNT)
            for (uint32_t i = tid; i < kFineBins; i += NT) sh.hist[i] = 0;
        const float ref = fixed_ref(b.st.cap, p);
        const RecStats rs = records_stats<false, kSmPer>(live, wm, nan, wsum, ref, want, sh.t, sh.c, dead);
        bool degenerate = rs.degenerate;
        double total = 0.0;
        if (part == 0 && !degenerate) {
            const double share = records_part<kSmPer>(wsum, wm, rs.gm, ref, sh.c.exp2_tbl);
            if (lane == 0) sh.c.redd[wave] = share;
            __syncthreads();
            for (int w = 0; w < NT / 64; ++w) total += sh.c.redd[w];
            degenerate = !(total > 0.0);  // sampling.cpp:116-118
        }
        if (part == 0 && tid == 0) {
            st.total = total;
            st.gm = rs.gm;
            st.scale = rs.scale;
            st.bstar = rs.bstar;
            st.degenerate = degenerate ? 1u : 0u;
        }
        if (degenerate) return;
        gm = rs.gm;
        scale = rs.scale;
        bstar = rs.bstar;
    } else {  // after the counting launch
        if (st.degenerate != 0) return;
        gm = st.gm;
        scale = st.scale;
        for (uint32_t i = tid; i < kFineBins; i += NT) sh.hist[i] = st.hist[i];
        if (tid == 0) sh.c.misc[3] = sh.c.misc[4] = 0;
        __syncthreads();
        fine_scan(sh.hist, sh.wsum);
        bstar = fine_bound(sh.hist, want, &sh.bound);
    }
    const double dgm = static_cast<double>(gm);
    RecStats coarse{};
    coarse.gm = gm;
    coarse.scale = scale;
    coarse.binned = scale != 0.0f;
    const FineBin fine = fine_bins(gm, scale, binned);
    const bool by_fine = !COUNT && binned;
    auto keep = [&](float v) {
        return (by_fine ? fine(v) : rec_bin(coarse, v)) <= bstar && !(static_cast<double>(v) - dgm < dead);
    };
    {
        bool is_cand[kSmPer];
        uint16_t id[kSmPer];
#pragma unroll
        for (uint32_t q = 0; q < kSmPer; ++q) {
            const uint32_t i = tid + NT * q;
            is_cand[q] = live[q] && i % parts == part && keep(wm[q]);
            id[q] = static_cast<uint16_t>(i);
        }
        wave_put_n(is_cand, id, &sh.c.misc[3], sh.cwave, kSampleMaxWaves);
    }
    __syncthreads();
    const uint32_t ncw = sh.c.misc[3];
    for_entries(sh.cwave, ncw, b.rec_shift, b.vocab, lg, [&](auto& v, auto& r, auto& in) {
        constexpr uint32_t N = sizeof(in) / sizeof(in[0]);
        bool kp[N];
        uint64_t kk[N];
#pragma unroll
        for (uint32_t q = 0; q < N; ++q) {
            kp[q] = in[q] && keep(v[q]);
            if constexpr (COUNT) {
                if (kp[q]) atomicAdd(&sh.hist[fine(v[q])], 1u);
            } else {
                kk[q] = kp[q] ? rank_key(v[q], r[q]) : 0ull;
            }
        }
        if constexpr (!COUNT) wave_put_n(kp, kk, &sh.c.misc[4], sh.keys, kPartCap);
    });
    __syncthreads();
    if constexpr (COUNT) {
        for (uint32_t i = tid; i < kFineBins; i += NT)
            if (sh.hist[i] != 0) atomicAdd(&st.hist[i], sh.hist[i]);
    } else {
        const uint32_t n = sh.c.misc[4];
        // a part that overflows makes the row's list one: the finish then gathers it again
        if (tid == 0 && n != 0) sh.base = atomicAdd(&st.n, n <= kPartCap ? n : kWideCap + 1);
        __syncthreads();
        if (n == 0 || n > kPartCap) return;
        uint64_t* keys = b.keys + static_cast<size_t>(j) * b.npad;
        for (uint32_t i = tid; i < n; i += NT)
            if (sh.base + i < kWideCap) keys[sh.base + i] = sh.keys[i];
    }
}

struct WideShared {
    union {
        uint64_t cand[kWideCap];  // the row's list
        struct {
            double e[kWideMax], q[kWideMax];  // then the shortlist's running sums
        } pre;
        LongFinishShared fin;
    } u;
    uint64_t sorted[kWideMax];
    union {
        uint16_t cwave[kSampleMaxWaves];  // candidate records, when the list is gathered again
        uint16_t order[kWideCap];         // then the list by fine bin
    } o;
    uint32_t hist[kFineBins];
    uint32_t wsum[16], lohi[2], big, cut, pick;
    TopScratch t;
    SelCommon c;
};
static_assert(sizeof(WideShared) <= 160 * 1024, "one block per CU");

// Counts into hist with a thread's two last bins held in registers: additions on one LDS address are
// served one after another, and a row that needs counting here is mostly one of few values.
struct Tally {
    uint32_t* hist;
    uint32_t b0 = 0, c0 = 0, b1 = 0, c1 = 0;
    __device__ __forceinline__ void add(uint32_t bin) {
        if (bin == b0) {
            ++c0;
        } else if (bin == b1) {
            ++c1;
        } else {
            if (c1 != 0) atomicAdd(&hist[b1], c1);
            b1 = b0;
            c1 = c0;
            b0 = bin;
            c0 = 1;
        }
    }
    __device__ __forceinline__ void flush() {
        if (c0 != 0) atomicAdd(&hist[b0], c0);
        if (c1 != 0) atomicAdd(&hist[b1], c1);
    }
};

// The smallest float that is not dead at a row maximum gm (see dead_distance): found next to the
// rounded sum, from where a step or two remain.
__device__ __forceinline__ float alive_floor(double gm, double dead) {
    if (dead == -INFINITY) return -INFINITY;
    auto alive = [&](uint32_t k) { return !(static_cast<double>(key_float(k)) - gm < dead); };
    uint32_t k = float_key(static_cast<float>(gm + dead));
    const uint32_t least = float_key(-INFINITY);
    while (!alive(k)) ++k;
    while (k > least && alive(k - 1)) --k;
    return key_float(k);
}

// The list of a row whose filters found more than kWideCap entries, by this block alone: the fine bins
// up to the want-th entry's, or where the last of them overflows too (ties, mostly), the ranks from a
// threshold up that leaves at most kWideCap. The threshold comes from counting that bin's entries by
// parts of its range of values, and where one value alone is too many, by ranges of index. Each pass
// reads the candidate records once, 16 entries a lane at a time, and is bound by its instructions per
// entry on the one CU; a row of equal entries takes four. A radix select of the want-th rank read them
// nine times, an entry at a time. The whole call, one row of V = 262,144, top_k = 300, us, with the
// long path, with the radix select, and now: equal entries 347, 1,389, 146; two values 348, 1,464, 266.
// Returns the list's length.
__device__ __forceinline__ uint32_t wide_regather(const LongBufs& b, const twd_row_params& p, uint32_t row, float gm,
                                                  const FineBin& fine, uint32_t want, WideShared& sh) {
    constexpr int NT = kLongThreads;
    constexpr uint32_t kRunShift = 4, kRun = 1u << kRunShift;
    const int tid = threadIdx.x;
    const uint32_t W = b.waves, rsh = b.rec_shift, vocab = b.vocab;
    const size_t o = static_cast<size_t>(row) * W;
    const float* lg = b.logits + static_cast<size_t>(row) * b.stride;
    const float floor = alive_floor(static_cast<double>(gm), wide_dead(p));
    auto list = [&](uint32_t bound) {  // records with an entry in a fine bin <= bound
        if (tid == 0) sh.c.misc[3] = sh.c.misc[4] = 0;
        __syncthreads();
        for (uint32_t i0 = 0; i0 < W; i0 += NT) {
            const uint32_t i = i0 + tid;
            const float m = i < W ? b.st.max[o + i] : -INFINITY;
            bool c[1] = {i < W && fine(m) <= bound && m >= floor};
            uint16_t id[1] = {static_cast<uint16_t>(i)};
            wave_put_n(c, id, &sh.c.misc[3], sh.o.cwave, kSampleMaxWaves);
        }
        __syncthreads();
    };
    // f(values, first row) over the listed records' entries, kRun consecutive ones a thread (a record
    // holds whole runs; their rows lie in one range of index); the same trip count in every thread.
    // Past the end NaN, which no comparison accepts.
    auto entries = [&](auto&& f) {
        const uint32_t esh = rsh - kRunShift, emask = (1u << esh) - 1u, ne = sh.c.misc[3] << esh;
        for (uint32_t i0 = 0; i0 < ne; i0 += NT) {
            const uint32_t e = i0 + tid;
            uint32_t r0 = vocab;
            if (e < ne) r0 = (static_cast<uint32_t>(sh.o.cwave[e >> esh]) << rsh) + ((e & emask) << kRunShift);
            float v[kRun];
            if (r0 + kRun <= vocab) {
#pragma unroll
                for (uint32_t q = 0; q < kRun / 4; ++q) {
                    const float4_u x = *reinterpret_cast<const float4_u*>(lg + r0 + 4 * q);
#pragma unroll
                    for (uint32_t k = 0; k < 4; ++k) v[4 * q + k] = x[k];
                }
            } else {
#pragma unroll
                for (uint32_t q = 0; q < kRun; ++q) v[q] = r0 + q < vocab ? lg[r0 + q] : __builtin_nanf("");
            }
            f(v, r0);
        }
        __syncthreads();
    };
    // the inclusive counts by bin(value, row) of the entries from lo to hi
    auto count = [&](float lo, float hi, auto&& bin) {
        for (uint32_t i = tid; i < kFineBins; i += NT) sh.hist[i] = 0;
        __syncthreads();
        Tally tally{sh.hist};
        entries([&](auto& v, uint32_t r) {
#pragma unroll
            for (uint32_t q = 0; q < kRun; ++q)
                if (v[q] >= lo && v[q] <= hi) tally.add(bin(v[q], r + q));
        });
        tally.flush();
        __syncthreads();
        fine_scan(sh.hist, sh.wsum);
    };
    auto gather = [&](auto&& keep) {
        entries([&](auto& v, uint32_t r) {
            bool kp[kRun];
            uint64_t kk[kRun];
#pragma unroll
            for (uint32_t q = 0; q < kRun; ++q) {
                kp[q] = keep(v[q], r + q);
                kk[q] = rank_key(v[q], r + q);
            }
            wave_put_n(kp, kk, &sh.c.misc[4], sh.u.cand, kWideCap);
        });
    };
    list(kFineBins - 1);
    count(floor, INFINITY, [&](float v, uint32_t) { return fine(v); });
    const uint32_t t = fine_bound(sh.hist, want, &sh.big);
    uint32_t n = sh.hist[t], above = t == 0 ? 0u : sh.hist[t - 1];  // up to the bin, and before it
    list(t);
    if (n <= kWideCap) {
        gather([&](float v, uint32_t) { return v >= floor && fine(v) <= t; });
        return n;
    }
    // the range of the bin's values
    if (tid == 0) {
        sh.lohi[0] = 0xFFFFFFFFu;
        sh.lohi[1] = 0u;
    }
    __syncthreads();
    {
        float lo = INFINITY, hi = -INFINITY;
        entries([&](auto& v, uint32_t) {
#pragma unroll
            for (uint32_t q = 0; q < kRun; ++q) {
                const bool in = v[q] >= floor && fine(v[q]) == t;
                lo = in ? fminf(lo, v[q]) : lo;
                hi = in ? fmaxf(hi, v[q]) : hi;
            }
        });
#pragma unroll
        for (int msk = 1; msk < 64; msk <<= 1) {
            lo = fminf(lo, __shfl_xor(lo, msk));
            hi = fmaxf(hi, __shfl_xor(hi, msk));
        }
        if ((tid & 63) == 0) {
            atomicMin(&sh.lohi[0], float_key(lo));
            atomicMax(&sh.lohi[1], float_key(hi));
        }
    }
    __syncthreads();
    uint32_t klo = sh.lohi[0], khi = sh.lohi[1];  // the list ends between these keys
    for (;;) {  // at most three ranges of values (2,048 parts each), then one value
        const bool one = klo == khi;
        const uint32_t span = one ? vocab - 1 : khi - klo;
        const uint32_t psh = span < kFineBins ? 0u : 21u - static_cast<uint32_t>(__builtin_clz(span));
        if (one)
            count(key_float(klo), key_float(khi), [&](float, uint32_t r) { return r >> psh; });
        else
            count(key_float(klo), key_float(khi), [&](float v, uint32_t) { return (khi - float_key(v)) >> psh; });
        const uint32_t part = fine_bound(sh.hist, want - above, &sh.big);
        const uint32_t before = part == 0 ? 0u : sh.hist[part - 1];
        n = above + sh.hist[part];
        const uint32_t end = min((part << psh) + ((1u << psh) - 1u), span);  // the part's last row or lowest key
        __syncthreads();  // the counts are read
        if (one) {  // above < want <= kWideMax, and a part has at most 256 rows: n < kWideCap
            const float x = key_float(khi);
            gather([&](float v, uint32_t r) { return v > x || (v == x && r <= end); });
            return n;
        }
        const uint32_t top = khi;
        khi = top - (part << psh);
        klo = top - end;
        if (n <= kWideCap) {
            const float x = key_float(klo);
            gather([&](float v, uint32_t) { return v >= x; });
            return n;
        }
        above += before;
    }
}

__global__ __launch_bounds__(kLongThreads) void wide_finish_kernel(LongArgs args_by_value, LongBufs b) {
    constexpr int NT = kLongThreads;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    WideShared& sh = *reinterpret_cast<WideShared*>(smem_raw);
    const LongArgs& args = TWD_LONG_ARGS(args_by_value);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t j = blockIdx.x;
    const uint32_t row = args.row[j];
    const twd_row_params p = args.p[j];
    const uint32_t want = min(static_cast<uint32_t>(p.top_k), b.vocab);  // <= kWideMax
    WideState& st = b.wide[j];
    const double total = st.total;
    const float gm = st.gm, scale = st.scale;
    const bool degenerate = st.degenerate != 0;
    uint32_t n = st.n;
    const uint64_t* list = b.keys + static_cast<size_t>(j) * b.npad;
    __syncthreads();  // every thread has read the state
    if (tid == 0) st.n = 0;
    if (wide_needs_bins(want, b.waves))
        for (uint32_t i = tid; i < kFineBins; i += NT) st.hist[i] = 0;
    if (degenerate) {
        if (tid == 0) b.tokens[row] = TWD_TOKEN_DEGENERATE;
        return;
    }
    FineBin fine = fine_bins(gm, scale, wide_needs_bins(want, b.waves));
    const double dgm = static_cast<double>(gm);
    if (n <= kWideCap) {
        for (uint32_t i = tid; i < kFineBins; i += NT) sh.hist[i] = 0;
        __syncthreads();
        for (uint32_t i = tid; i < n; i += NT) {
            const uint64_t k = list[i];
            sh.u.cand[i] = k;
            atomicAdd(&sh.hist[fine(rank_value(k))], 1u);
        }
        __syncthreads();
        fine_scan(sh.hist, sh.wsum);
    } else {
        n = wide_regather(b, p, row, gm, fine, want, sh);
        for (uint32_t i = tid; i < kFineBins; i += NT) sh.hist[i] = 0;
        __syncthreads();
        for (uint32_t i = tid; i < n; i += NT) atomicAdd(&sh.hist[fine(rank_value(sh.u.cand[i]))], 1u);
        __syncthreads();
        fine_scan(sh.hist, sh.wsum);
    }

    // ---- sorted[0 .. nl): the shortlist's live entries in descending order
    const uint32_t nl = min(n, want);
    const uint32_t below = sh.hist[kFineBins - 2];
    if (below < nl && n - below > kWideLast) {
        // The last bin holds what lies past the records' range, which is much of a small vocabulary taken
        // whole: bins over the list's own range instead. Whole call, us, the long path before these
        // kernels, without this, with it: V = 300, top_k = 300, one row 33.2, 38.6, 29.4; V = 1,500,
        // top_k = 4,096, 64 rows 54.6, 60.7, 36.3.
        if (tid == 0) sh.lohi[0] = 0xFFFFFFFFu;
        __syncthreads();  // also: the counts are read
        uint32_t least = 0xFFFFFFFFu;
        for (uint32_t i = tid; i < n; i += NT) least = min(least, static_cast<uint32_t>(sh.u.cand[i] >> 32));
#pragma unroll
        for (int msk = 1; msk < 64; msk <<= 1)
            least = min(least, static_cast<uint32_t>(__shfl_xor(static_cast<int>(least), msk)));
        if (lane == 0) atomicMin(&sh.lohi[0], least);
        for (uint32_t i = tid; i < kFineBins; i += NT) sh.hist[i] = 0;
        __syncthreads();
        const float span = gm - key_float(sh.lohi[0]);  // infinite: one bin
        fine.scale = static_cast<float>(kFineBins - 1) / span;
        for (uint32_t i = tid; i < n; i += NT) atomicAdd(&sh.hist[fine(rank_value(sh.u.cand[i]))], 1u);
        __syncthreads();
        fine_scan(sh.hist, sh.wsum);
    }
    if (tid == 0) sh.big = 0;
    __syncthreads();
    uint32_t lo[2];  // the starts of this thread's two bins
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const uint32_t i = 2 * tid + q;
        lo[q] = i == 0 ? 0u : sh.hist[i - 1];
        if (lo[q] < nl && sh.hist[i] - lo[q] > kWideBucket) sh.big = 1;  // every writer writes 1
    }
    __syncthreads();
    if (sh.big == 0) {
#pragma unroll
        for (int q = 0; q < 2; ++q) sh.hist[2 * tid + q] = lo[q];
        __syncthreads();
        for (uint32_t i = tid; i < n; i += NT)
            sh.o.order[atomicAdd(&sh.hist[fine(rank_value(sh.u.cand[i]))], 1u)] = static_cast<uint16_t>(i);
        __syncthreads();  // hist[b] is bin b's end again
        for (uint32_t i = tid; i < n; i += NT) {
            const uint64_t k = sh.u.cand[i];
            const uint32_t bin = fine(rank_value(k));
            const uint32_t s0 = bin == 0 ? 0u : sh.hist[bin - 1], s1 = sh.hist[bin];
            if (s0 >= nl) continue;
            uint32_t at = s0;
            for (uint32_t s = s0; s < s1; s += 4) {  // four at a time: each is two LDS reads in a row
                uint16_t e[4];
                uint64_t o[4];
#pragma unroll
                for (uint32_t q = 0; q < 4; ++q) e[q] = sh.o.order[min(s + q, s1 - 1)];
#pragma unroll
                for (uint32_t q = 0; q < 4; ++q) o[q] = sh.u.cand[e[q]];
#pragma unroll
                for (uint32_t q = 0; q < 4; ++q) at += s + q < s1 && o[q] > k ? 1u : 0u;
            }
            if (at < nl) sh.sorted[at] = k;
        }
    } else {
        uint32_t len = 2;
        while (len < n) len <<= 1;  // <= kWideCap
        for (uint32_t i = n + tid; i < len; i += NT) sh.u.cand[i] = 0ull;
        __syncthreads();
        for (uint32_t k = 2; k <= len; k <<= 1) bitonic_tile_steps(sh.u.cand, len, 0, k, k >> 1);
        for (uint32_t i = tid; i < nl; i += NT) sh.sorted[i] = sh.u.cand[i];
    }
    __syncthreads();

    // ---- steps 5-7: running sums of the terms (sampling.cpp:145,157), `tpt` consecutive per thread
    const double td = static_cast<double>(p.temperature), pp = static_cast<double>(p.top_p);
    const bool topp = p.top_p < 1.0f;
    constexpr uint32_t kTpt = kWideMax / NT;
    const uint32_t tpt = (want + NT - 1) / NT, i0 = tid * tpt;
    double pe[kTpt], pq[kTpt], se = 0.0, sq = 0.0;
#pragma unroll
    for (uint32_t q = 0; q < kTpt; ++q) {
        pe[q] = pq[q] = 0.0;
        if (q < tpt && i0 + q < nl) {
            const double l = static_cast<double>(rank_value(sh.sorted[i0 + q]));
            pq[q] = exp_libm((l - dgm) / td);
            if (topp) pe[q] = exp_libm(l - dgm) / total;
        }
        se += pe[q];
        sq += pq[q];
        pe[q] = se;
        pq[q] = sq;
    }
    const double we = wave_incl_scan_f64(se), wq = wave_incl_scan_f64(sq);
    if (lane == 63) {
        sh.c.redd[wave] = we;
        sh.c.e[wave] = wq;
    }
    if (tid == 0) {
        sh.cut = want;
        sh.pick = want;
    }
    __syncthreads();
    double ae = 0.0, aq = 0.0;  // the waves and the lanes below
    for (int w = 0; w < wave; ++w) {
        ae += sh.c.redd[w];
        aq += sh.c.e[w];
    }
    ae += dpp_move<0x138>(0.0, we);
    aq += dpp_move<0x138>(0.0, wq);
#pragma unroll
    for (uint32_t q = 0; q < kTpt; ++q)
        if (q < tpt && i0 + q < want) {
            sh.u.pre.e[i0 + q] = ae + pe[q];
            sh.u.pre.q[i0 + q] = aq + pq[q];
        }
    __syncthreads();
    // the first prefix that reaches x (one writer where the prefixes rise; where rounding makes
    // them fall by an ulp, x lies within the margin)
    auto first = [&](const double* pre, uint32_t lim, double x, uint32_t* out) {
        for (uint32_t i = tid; i < lim; i += NT)
            if (pre[i] >= x && (i == 0 || pre[i - 1] < x)) atomicMin(out, i);
        __syncthreads();
        return *out;
    };
    bool ok = true;
    uint32_t cut = want;
    if (topp) {
        const double tc = kSumTol + total_tol(b.vocab);
        const uint32_t i = first(sh.u.pre.e, want, pp, &sh.cut);
        if (i < want) {
            cut = i + 1;
            ok = sh.u.pre.e[i] >= pp * (1.0 + tc) && (i == 0 || sh.u.pre.e[i - 1] < pp * (1.0 - tc));
        } else {
            ok = sh.u.pre.e[want - 1] < pp * (1.0 - tc);
        }
    }
    const double r = static_cast<double>(p.uniform) * sh.u.pre.q[cut - 1];
    const uint32_t pick = first(sh.u.pre.q, cut, r, &sh.pick);
    if (pick < cut)
        ok = ok && sh.u.pre.q[pick] >= r * (1.0 + kSumTol) &&
             (pick == 0 || sh.u.pre.q[pick - 1] < r * (1.0 - kSumTol));
    else
        ok = false;
    if (ok && pick < nl) {
        if (tid == 0) b.tokens[row] = rank_index(sh.sorted[pick]);
        return;
    }
    // within the margin (the same in every thread): the reference's own sums, from memory. Dead
    // entries stand in as ranks of -inf, whose terms are 0.
    uint64_t* keys = b.keys + static_cast<size_t>(j) * b.npad;
    for (uint32_t i = tid; i < want; i += NT) keys[i] = i < nl ? sh.sorted[i] : rank_key(-INFINITY, 0);
    __syncthreads();
    long_finish_row_call(args, b, j, gm, total, sh.u.fin);
}

// ---- the wave-record path for logits that are already in memory ---------------------------------
//
// Rows whose logits the caller holds (twd_select, the head for rows > 4) reach
// select_sample_merge_kernel through two short passes instead of the slice kernels:
//   * penalty_hash_kernel, one block per row: the row's history ids into an LDS hash table of
//     (id, occurrences) while each id's logit is requested, then each distinct id's logit gets
//     the penalty once per occurrence, one after another as the reference loop applies them
//     (sampling.cpp:74-90), from the thread that entered the id; only those entries are read
//     and written;
//   * wave_stats_kernel: per 64 entries of a row, the record the head's sample mode publishes
//     -- the best rank (value desc, index asc) and the sum of exp(v - that value) in double,
//     NaN when a NaN was seen. Eight lanes hold one record's 64 entries, eight each.
constexpr int kPhThreads = 1024;
constexpr uint32_t kHashSlots = 8192;    // LDS hash table of one row's history
constexpr uint32_t kHashMaxIds = 4096;   // history ids per row the table takes (load <= 1/2)
constexpr uint32_t kHashEmpty = 0xFFFFFFFFu;  // never an id below vocab <= 2^30

struct PenaltyBufs {
    float* logits;
    uint64_t stride;
    uint32_t vocab;
    const uint32_t* history;
};

__global__ __launch_bounds__(kPhThreads) void penalty_hash_kernel(SelectArgs args_by_value, PenaltyBufs b) {
    constexpr int NT = kPhThreads;
    constexpr uint32_t kIdsPer = kHashMaxIds / NT;     // history ids per thread
    constexpr uint32_t kSlotsPer = kHashSlots / NT;    // table slots per thread
    __shared__ uint32_t keys[kHashSlots];
    __shared__ uint32_t cnt[kHashSlots];
#if __HIP_DEVICE_COMPILE__
    const SelectArgs& args =
        *reinterpret_cast<const SelectArgs*>(__builtin_amdgcn_kernarg_segment_ptr());
#else
    const SelectArgs& args = args_by_value;
#endif
    const int tid = threadIdx.x;
    const uint32_t row = blockIdx.x;
    const twd_row_params p = args.p[row];
    if (p.repetition_penalty == 1.0f || p.history_len == 0) return;  // the whole block
    // every id requested at once (history_len <= kHashMaxIds, checked by the launch)
    const uint32_t* hist = b.history + p.history_offset;
    uint32_t ids[kIdsPer];
#pragma unroll
    for (uint32_t q = 0; q < kIdsPer; ++q) {
        const uint32_t j = tid + NT * q;
        const uint32_t id = hist[min(j, p.history_len - 1)];  // unconditional: no branch per load
        ids[q] = j < p.history_len ? id : kHashEmpty;
    }
#pragma unroll
    for (uint32_t q = 0; q < kSlotsPer; ++q) {
        keys[tid + NT * q] = kHashEmpty;
        cnt[tid + NT * q] = 0;
    }
    // each id's logit, requested now so that its round trip overlaps the table's construction
    // (only the thread that enters an id into the table uses it)
    float* lg = b.logits + static_cast<size_t>(row) * b.stride;
    float x[kIdsPer];
#pragma unroll
    for (uint32_t q = 0; q < kIdsPer; ++q) x[q] = lg[ids[q] < b.vocab ? ids[q] : 0u];  // no branch per load
    __syncthreads();
    uint32_t slot[kIdsPer];  // the slot this thread entered id q into, or kHashEmpty
#pragma unroll
    for (uint32_t q = 0; q < kIdsPer; ++q) {
        const uint32_t id = ids[q];
        slot[q] = kHashEmpty;
        if (id >= b.vocab) continue;  // out-of-range ids are ignored (sampling.cpp:82)
        // linear probing from a multiplicative hash; the table is at most half full, so a free
        // or matching slot is always found
        uint32_t h = (id * 0x9E3779B1u) >> (32 - 13);
        for (;;) {
            const uint32_t prev = atomicCAS(&keys[h], kHashEmpty, id);
            if (prev == kHashEmpty || prev == id) {
                atomicAdd(&cnt[h], 1u);
                if (prev == kHashEmpty) slot[q] = h;
                break;
            }
            h = (h + 1) & (kHashSlots - 1);
        }
    }
    __syncthreads();
    const float rp = p.repetition_penalty;
    const float limit = (p.softcap > 0.0f) ? p.softcap * 0.9999f : 0.0f;
    // each distinct id, by the thread that entered it: the penalty once per occurrence, the store
#pragma unroll
    for (uint32_t q = 0; q < kIdsPer; ++q) {
        if (slot[q] == kHashEmpty) continue;
        const uint32_t n = cnt[slot[q]];
        float v = x[q];
        for (uint32_t t = 0; t < n; ++t) {
            v = (v > 0.0f) ? (v / rp) : (v * rp);
            if (limit > 0.0f) v = (v < -limit) ? -limit : ((limit < v) ? limit : v);
        }
        lg[ids[q]] = v;
    }
}

// NB 8-entry batches per lane. One: many short blocks, so that later blocks' loads overlap
// earlier blocks' arithmetic (with four, every wave requested all its loads first, and the pass
// ran as a load phase, then an arithmetic phase).
template <uint32_t NB, bool AUX>
__global__ __launch_bounds__(kWsThreads) __attribute__((amdgpu_waves_per_eu(8)))
void wave_stats_kernel(WaveStatsBufs b) {
    __shared__ double tbl[64];
    wave_records_block<NB, AUX>(b, blockIdx.x, blockIdx.y, tbl);
}

// When the record pass also forms the record words: for few rows, whose blocks are short of work,
// and for long shortlists, whose merges they spare the most gathering. The words cost the pass time by
// the entries of all rows, and a merge is spared time by its own shortlist (from 128 entries on, where it
// gathers in more batches), so the mean shortlist past 64 is held against the entries. Without the words
// and with them, us: 48 rows of V = 32,003 k = 128 15.9 and 15.9, k = 256 22.2 and 19.1; of 151,669 k = 128
// 22.9 and 22.2, k = 256 28.2 and 25.2; of 262,144 k = 64 24.3 and 26.4, k = 128 27.4 and 27.7, k = 200 29.4 and 28.8;
// 64 rows of 262,144 k = 128 30.8 and 31.7, k = 256 36.2 and 34.4; of 500,000 k = 128 46.7 and 49.6, k = 200
// 48.5 and 50.7.
constexpr uint32_t kAuxMaxRows = 8;
constexpr uint32_t kAuxMeanWant = 128;

static bool want_aux(uint32_t rows, uint32_t vocab, uint32_t want_sum) {
    if (rows <= kAuxMaxRows) return true;
    if (want_sum < kAuxMeanWant * rows) return false;
    return static_cast<uint64_t>(rows) * rows * vocab <= 160000ull * (want_sum - 64ull * rows);
}

__global__ void verify_compare_kernel(const uint32_t* row_tokens, uint32_t rows,
                                      const uint32_t* drafts, uint32_t nd,
                                      twd_verify_result* v) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    uint32_t n = 0, acc = 0, bonus = 0, sampled = 0;
    bool bad = false;
    if (nd != 0 && rows != 0) {
        const uint32_t k = nd < rows ? nd : rows;
        bool rejected = false;
        for (uint32_t i = 0; i < k; ++i) {
            const uint32_t t = row_tokens[i];
            if (t == TWD_TOKEN_DEGENERATE) {
                bad = true;
                break;
            }
            if (drafts[i] == t) {
                v->tokens[n++] = t;
                ++acc;
            } else {
                bonus = t;
                sampled = 1;
                v->tokens[n++] = t;
                rejected = true;
                break;
            }
        }
        if (!bad && !rejected && rows > k) {
            bonus = row_tokens[k];
            if (bonus == TWD_TOKEN_DEGENERATE) bad = true;
            sampled = 1;
            v->tokens[n++] = bonus;
        }
    }
    v->n_tokens = bad ? TWD_TOKEN_DEGENERATE : n;
    v->num_accepted = acc;
    v->total_drafted = nd;
    v->bonus_token_sampled = sampled;
    v->bonus_token = bonus;
}

// ---- scratch and launch helpers ----------------------------------------------------------------

static uint32_t parts_for(uint32_t vocab) { return (vocab + kSlice - 1) / kSlice; }

// ---- the no-allocation selection: scratch in a device array of fixed size ------------------------
// The selection scratch of at most kStaticRows rows of at most kStaticVocab entries, carved the
// way scratch_alloc lays it out. Each GPU holds its own copy for the life of the process; every
// twd_select_noalloc call on a GPU shares it.
constexpr uint32_t kStaticRows = TWD_MAX_ROWS;
constexpr uint32_t kStaticVocab = 262144;
constexpr uint32_t kStaticParts = kStaticVocab / kSlice;  // 32
constexpr size_t kStaticSlots = static_cast<size_t>(kStaticRows) * kStaticParts;
constexpr size_t kStaticOffSum = 0;                                   // double [slots]
constexpr size_t kStaticOffKey = kStaticOffSum + 8 * kStaticSlots;    // uint64 [slots]
constexpr size_t kStaticOffMax = kStaticOffKey + 8 * kStaticSlots;    // float [slots]
constexpr size_t kStaticOffFlag = kStaticOffMax + 4 * kStaticSlots;   // uint32 [slots]
constexpr size_t kStaticOffCount = kStaticOffFlag + 4 * kStaticSlots; // uint32 [slots]
constexpr size_t kStaticOffCand = kStaticOffCount + 4 * kStaticSlots; // uint64 [slots][kMaxWant]
constexpr size_t kStaticOffGbest = kStaticOffCand + 8 * kStaticSlots * kMaxWant;  // uint64 [rows + kArriveWords]
constexpr size_t kStaticBytes = kStaticOffGbest + 8 * (kStaticRows + kArriveWords);  // 4,252,208 B
static_assert(kStaticBytes == 4252208, "the size twd_head.h states");
static_assert(kStaticOffCand % 256 == 0, "candidate array alignment");

static __device__ __align__(256) unsigned char scratch[kStaticBytes];

namespace {

// The device address of `scratch` on each GPU (its own copy there), found once per device with
// that device current. Host code uses these addresses, never the array's name: on the host the
// name is a stand-in that no kernel may dereference.
constexpr int kMaxDevices = 64;
std::mutex g_static_mu;
void* g_static_ptr[kMaxDevices] = {};
uint32_t g_static_epoch[kMaxDevices] = {};  // of each GPU's last one-pass greedy launch

int static_scratch(SelectScratch* out) {
    int dev = 0;
    TWD_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(TWD_E_UNSUPPORTED, "device index above 63");
    void* base = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_static_mu);
        if (!g_static_ptr[dev]) {
            void* p = nullptr;
            TWD_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
            if (!p) return fail(TWD_E_HIP, "hipGetSymbolAddress returned no address for the scratch array");
            g_static_ptr[dev] = p;
        }
        base = g_static_ptr[dev];
    }
    unsigned char* b = static_cast<unsigned char*>(base);
    SelectScratch s{};
    s.max_rows = kStaticRows;
    s.max_parts = kStaticParts;
    s.part_sum = reinterpret_cast<double*>(b + kStaticOffSum);
    s.part_key = reinterpret_cast<uint64_t*>(b + kStaticOffKey);
    s.part_max = reinterpret_cast<float*>(b + kStaticOffMax);
    s.part_flag = reinterpret_cast<uint32_t*>(b + kStaticOffFlag);
    s.part_count = reinterpret_cast<uint32_t*>(b + kStaticOffCount);
    s.cand = reinterpret_cast<uint64_t*>(b + kStaticOffCand);
    // zero at load: the first one-pass greedy launch on a GPU finds the counter unarmed and
    // counts in on the fallback word, then arms it for the next
    s.gbest = reinterpret_cast<uint64_t*>(b + kStaticOffGbest);
    s.gctr = s.gbest + kStaticRows;
    s.epoch = &g_static_epoch[dev];
    s.verify_tokens = nullptr;  // twd_select does not use it
    *out = s;
    return TWD_OK;
}

}  // namespace

int scratch_alloc(SelectScratch* s, uint32_t max_vocab, uint32_t max_rows) {
    s->max_rows = max_rows;
    s->max_parts = parts_for(max_vocab);
    const size_t n = static_cast<size_t>(max_rows) * s->max_parts;
    hipError_t e = hipSuccess;
    if (e == hipSuccess) e = hipMalloc(&s->part_max, n * sizeof(float));
    if (e == hipSuccess) e = hipMalloc(&s->part_sum, n * sizeof(double));
    if (e == hipSuccess) e = hipMalloc(&s->part_flag, n * sizeof(uint32_t));
    if (e == hipSuccess) e = hipMalloc(&s->part_count, n * sizeof(uint32_t));
    if (e == hipSuccess) e = hipMalloc(&s->part_key, n * sizeof(uint64_t));
    if (e == hipSuccess) e = hipMalloc(&s->cand, n * kMaxWant * sizeof(uint64_t));
    if (e == hipSuccess) e = hipMalloc(&s->verify_tokens, (max_rows + 1) * sizeof(uint32_t));
    // the wave records of the wave-record path, ceil(max_vocab / 64) per row
    s->wave_cap = (max_vocab + kSampleWaveRows - 1) / kSampleWaveRows;
    const size_t nw = static_cast<size_t>(max_rows) * s->wave_cap;
    if (e == hipSuccess) e = hipMalloc(&s->wkey, nw * sizeof(uint64_t));
    if (e == hipSuccess) e = hipMalloc(&s->wsum, nw * sizeof(double));
    if (e == hipSuccess) e = hipMalloc(&s->wmax, nw * sizeof(float));
    if (e == hipSuccess) e = hipMalloc(&s->waux, nw * sizeof(uint32_t));
    if (e == hipSuccess) e = hipMalloc(&s->gbest, (max_rows + kArriveWords) * sizeof(uint64_t));
    if (e == hipSuccess) e = hipMemset(s->gbest, 0, (max_rows + kArriveWords) * sizeof(uint64_t));
    const uint64_t armed = kFirstEpoch;  // the counter starts armed for the first launch
    if (e == hipSuccess) e = hipMemcpy(s->gbest + max_rows, &armed, sizeof(armed), hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        s->gctr = s->gbest + max_rows;
        s->epoch = new uint32_t(kFirstEpoch - 1);
        s->lng = new LongScratch();
    }
    if (e != hipSuccess) {
        scratch_free(s);
        return hip_fail(e, "allocating selection scratch");
    }
    return TWD_OK;
}

void scratch_free(SelectScratch* s) {
    (void)hipFree(s->part_max);
    (void)hipFree(s->part_sum);
    (void)hipFree(s->part_flag);
    (void)hipFree(s->part_count);
    (void)hipFree(s->part_key);
    (void)hipFree(s->cand);
    (void)hipFree(s->verify_tokens);
    (void)hipFree(s->wkey);
    (void)hipFree(s->wsum);
    (void)hipFree(s->wmax);
    (void)hipFree(s->waux);
    (void)hipFree(s->gbest);
    delete s->epoch;
    if (s->lng) {
        long_free(s->lng);
        delete s->lng;
    }
    *s = SelectScratch{};
}

void long_free(LongScratch* l) {
    (void)hipFree(l->block);
    for (uint32_t i = 0; i < l->n_retired; ++i) (void)hipFree(l->retired[i]);
    *l = LongScratch{};
}

namespace {
// Zeroes device memory now, on a stream of its own: the caller's is under capture.
hipError_t zero_now(void* p, size_t bytes) {
    hipStream_t side = nullptr;
    hipError_t e = hipStreamCreateWithFlags(&side, hipStreamNonBlocking);
    if (e != hipSuccess) return e;
    e = hipMemsetAsync(p, 0, bytes, side);
    if (e == hipSuccess) e = hipStreamSynchronize(side);
    (void)hipStreamDestroy(side);
    return e;
}

int long_reserve(LongScratch* l, uint32_t rows, uint64_t npad, hipStream_t stream) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    TWD_HIP(hipStreamIsCapturing(stream, &cap));
    const bool capturing = cap != hipStreamCaptureStatusNone;
    if (l->block && l->rows_cap >= rows && l->npad_cap >= npad) {
        l->captured |= capturing;
        return TWD_OK;
    }
    uint32_t r = std::max(rows, l->rows_cap);
    const uint64_t n = std::max(npad, l->npad_cap);
    if (l->captured) {
        if (l->n_retired == sizeof(l->retired) / sizeof(l->retired[0]))
            return fail(TWD_E_UNSUPPORTED, "the long-shortlist scratch has outgrown too many captures");
        if (rows > l->rows_cap) r = std::max(rows, std::min(2 * l->rows_cap, static_cast<uint32_t>(TWD_MAX_ROWS)));
        l->retired[l->n_retired++] = l->block;
    } else {
        (void)hipFree(l->block);  // waits for the device before the old buffers go
    }
    l->block = nullptr;
    l->rows_cap = 0;
    l->npad_cap = 0;
    l->captured = capturing;
    const size_t m = static_cast<size_t>(r) * n;
    size_t bytes = 0;
    auto place = [&](size_t size) {
        const size_t at = bytes;
        bytes += (size + 255) / 256 * 256;
        return at;
    };
    const size_t keys = place(m * sizeof(uint64_t)), pre = place(m * sizeof(double)), len = place(r * sizeof(uint32_t)),
                 gmax = place(r * sizeof(float)), total = place(r * sizeof(double)), wide = place(r * sizeof(WideState));
    hipError_t e = hipMalloc(&l->block, bytes);
    char* const base = static_cast<char*>(l->block);
    if (e == hipSuccess) {
        // captured, the clear would only run with the replays, after eager calls that need it
        e = capturing ? zero_now(base + wide, r * sizeof(WideState))
                      : hipMemsetAsync(base + wide, 0, r * sizeof(WideState), stream);
    }
    if (e != hipSuccess) {
        (void)hipFree(l->block);
        l->block = nullptr;
        return hip_fail(e, "allocating the long-shortlist scratch");
    }
    l->keys = reinterpret_cast<uint64_t*>(base + keys);
    l->pre = reinterpret_cast<double*>(base + pre);
    l->len = reinterpret_cast<uint32_t*>(base + len);
    l->gmax = reinterpret_cast<float*>(base + gmax);
    l->total = reinterpret_cast<double*>(base + total);
    l->wide = reinterpret_cast<WideState*>(base + wide);
    l->rows_cap = r;
    l->npad_cap = n;
    return TWD_OK;
}
}  // namespace

int launch_long(LongScratch* lng, const SampleStats& st, uint32_t waves, uint32_t rec_rows, const float* logits,
                uint64_t stride, uint32_t vocab, uint32_t rows, const twd_row_params* params, uint32_t* tokens,
                hipStream_t stream) {
    LongArgs a{}, w{};  // shortlists past kWideMax, and up to it
    for (uint32_t r = 0; r < rows; ++r) {
        if (!long_row(params[r], vocab)) continue;
        LongArgs& x = std::min(static_cast<uint32_t>(params[r].top_k), vocab) <= kWideMax ? w : a;
        x.row[x.n] = r;
        x.p[x.n] = params[r];
        ++x.n;
    }
    if (a.n == 0 && w.n == 0) return TWD_OK;
    if (!lng) return fail(TWD_E_INVALID, "top_k > 256 needs a selector's scratch (twd_select)");
    if (waves == 0 || waves > kSampleMaxWaves) return fail(TWD_E_INVALID, "long shortlist: wave records out of range");
    uint64_t npad = kWideCap;
    while (npad < vocab) npad <<= 1;
    const int rc = long_reserve(lng, a.n + w.n, npad, stream);
    if (rc) return rc;
    LongBufs b{};
    b.logits = logits;
    b.stride = stride;
    b.vocab = vocab;
    b.waves = waves;
    b.rec_shift = static_cast<uint32_t>(__builtin_ctz(rec_rows));
    b.st = st;
    b.npad = npad;
    b.keys = lng->keys;
    b.pre = lng->pre;
    b.len = lng->len;
    b.gmax = lng->gmax;
    b.total = lng->total;
    b.wide = lng->wide;
    b.tokens = tokens;
    if (w.n != 0) {
        // enough parts to spread the rows' entries over the chip, few enough that their own passes
        // over the records stay a small part of the work
        const uint32_t parts = std::min(32u, std::max(4u, 256u / w.n));
        bool bins = false;
        for (uint32_t j = 0; j < w.n; ++j)
            bins |= wide_needs_bins(std::min(static_cast<uint32_t>(w.p[j].top_k), vocab), waves);
        if (bins) {
            wide_filter_kernel<true><<<dim3(parts, w.n), kLongThreads, sizeof(WideFilterShared), stream>>>(w, b);
            TWD_HIP(hipGetLastError());
        }
        wide_filter_kernel<false><<<dim3(parts, w.n), kLongThreads, sizeof(WideFilterShared), stream>>>(w, b);
        TWD_HIP(hipGetLastError());
        wide_finish_kernel<<<w.n, kLongThreads, sizeof(WideShared), stream>>>(w, b);
        TWD_HIP(hipGetLastError());
    }
    if (a.n == 0) return TWD_OK;
    long_gather_kernel<<<a.n, kLongThreads, sizeof(LongGatherShared), stream>>>(a, b);
    TWD_HIP(hipGetLastError());
    const uint32_t tile = static_cast<uint32_t>(std::min<uint64_t>(npad, kSortTile));
    const size_t tile_bytes = static_cast<size_t>(tile) * sizeof(uint64_t);
    const uint32_t ntile = static_cast<uint32_t>(npad / tile);
    long_sort_tile_kernel<<<dim3(ntile, a.n), kLongThreads, tile_bytes, stream>>>(b, tile);
    TWD_HIP(hipGetLastError());
    for (uint64_t k = 2ull * tile; k <= npad; k <<= 1) {
        for (uint64_t jj = k >> 1; jj >= tile; jj >>= 1) {
            long_sort_step_kernel<<<dim3(static_cast<uint32_t>(npad / 2 / kStepThreads), a.n), kStepThreads, 0,
                                    stream>>>(b, static_cast<uint32_t>(k), static_cast<uint32_t>(jj));
            TWD_HIP(hipGetLastError());
        }
        long_sort_merge_kernel<<<dim3(ntile, a.n), kLongThreads, tile_bytes, stream>>>(b, tile,
                                                                                       static_cast<uint32_t>(k));
        TWD_HIP(hipGetLastError());
    }
    long_finish_kernel<<<a.n, kLongThreads, 0, stream>>>(a, b);
    TWD_HIP(hipGetLastError());
    return TWD_OK;
}

// Lets the selection kernels use the LDS they need (no memory is allocated).
int enable_select_kernels() {
    static std::once_flag once;
    static hipError_t err = hipSuccess;
    std::call_once(once, [] {
        err = hipFuncSetAttribute(reinterpret_cast<const void*>(select_slice_kernel),
                                  hipFuncAttributeMaxDynamicSharedMemorySize,
                                  static_cast<int>(sizeof(SliceShared)));
        if (err == hipSuccess)
            err = hipFuncSetAttribute(reinterpret_cast<const void*>(select_merge_kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize,
                                      static_cast<int>(sizeof(MergeShared)));
        for (uint32_t waves : {1u, kSmThreads + 1u, 2 * kSmThreads + 1u, kSampleMaxWaves})
            for (MergeKernel merge : {merge_kernel<4>(waves), merge_kernel<5>(waves), merge_kernel<6>(waves)})
                if (err == hipSuccess && merge)
                    err = hipFuncSetAttribute(reinterpret_cast<const void*>(merge),
                                              hipFuncAttributeMaxDynamicSharedMemorySize,
                                              static_cast<int>(sizeof(SampleMergeShared)));
        if (err == hipSuccess)
            err = hipFuncSetAttribute(reinterpret_cast<const void*>(long_gather_kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize,
                                      static_cast<int>(sizeof(LongGatherShared)));
        if (err == hipSuccess)
            err = hipFuncSetAttribute(reinterpret_cast<const void*>(wide_filter_kernel<false>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize,
                                      static_cast<int>(sizeof(WideFilterShared)));
        if (err == hipSuccess)
            err = hipFuncSetAttribute(reinterpret_cast<const void*>(wide_filter_kernel<true>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize,
                                      static_cast<int>(sizeof(WideFilterShared)));
        if (err == hipSuccess)
            err = hipFuncSetAttribute(reinterpret_cast<const void*>(wide_finish_kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize,
                                      static_cast<int>(sizeof(WideShared)));
        if (err == hipSuccess)
            err = hipFuncSetAttribute(reinterpret_cast<const void*>(long_sort_tile_kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize,
                                      static_cast<int>(kSortTile * sizeof(uint64_t)));
        if (err == hipSuccess)
            err = hipFuncSetAttribute(reinterpret_cast<const void*>(long_sort_merge_kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize,
                                      static_cast<int>(kSortTile * sizeof(uint64_t)));
    });
    if (err != hipSuccess) return hip_fail(err, "hipFuncSetAttribute(MaxDynamicSharedMemorySize)");
    return TWD_OK;
}

int launch_select(const SelectScratch& s, float* logits, uint32_t vocab, uint32_t rows,
                  uint64_t stride, const twd_row_params* params, const uint32_t* history,
                  uint32_t* tokens, hipStream_t stream, bool penalty_only) {
    if (!logits || !params || (!tokens && !penalty_only))
        return fail(TWD_E_INVALID, "null logits, tokens or params");
    if (vocab == 0) return fail(TWD_E_INVALID, "sample_token: empty vocabulary");
    if (rows == 0 || rows > s.max_rows) return fail(TWD_E_INVALID, "rows out of range for this selector");
    const uint32_t parts = parts_for(vocab);
    if (parts > s.max_parts || parts > kMaxParts) return fail(TWD_E_INVALID, "vocab larger than this selector's max_vocab");
    if (stride < vocab) return fail(TWD_E_INVALID, "row_stride < vocab");
    SelectArgs a{};
    a.rows = rows;
    a.parts = parts;
    a.penalty_only = penalty_only ? 1u : 0u;
    bool any_long = false, any_short = false;  // any_short: a row that the merge finishes
    uint32_t short_want = 0;                   // the sampled ones' shortlists together
    for (uint32_t r = 0; r < rows; ++r) {
        const twd_row_params& p = params[r];
        if (p.repetition_penalty != 1.0f && p.history_len > 0 && !history)
            return fail(TWD_E_INVALID, "null history with a non-empty history_len");
        a.p[r] = p;
        any_long |= !penalty_only && long_row(p, vocab);
        any_short |= !long_row(p, vocab);
        if (!long_row(p, vocab) && !(p.temperature <= 0.0f))
            short_want += p.top_k > 0 ? static_cast<uint32_t>(p.top_k) : kMaxWant;
    }
    const uint32_t waves = (vocab + kSampleWaveRows - 1) / kSampleWaveRows;
    const bool have_records = s.wkey != nullptr && waves <= s.wave_cap && waves <= kSampleMaxWaves;
    if (any_long && (!s.lng || !have_records))
        return fail(TWD_E_INVALID, "top_k > 256 needs a selector's scratch (twd_select, not twd_select_noalloc)");
    // sampled rows with short histories: the wave-record path (penalty pass, per-64-entry
    // statistics, then the one-block-per-row merge that reads only the candidate waves)
    bool records = !penalty_only && have_records;
    bool any_sampled = false, any_penalty = false;
    for (uint32_t r = 0; r < rows; ++r) {
        const twd_row_params& p = params[r];
        any_sampled |= !(p.temperature <= 0.0f);
        if (p.repetition_penalty != 1.0f && p.history_len > 0) {
            any_penalty = true;
            records &= p.history_len <= kHashMaxIds;
        }
    }
    if (records && any_sampled) {
        int rc = enable_select_kernels();
        if (rc) return rc;
        if (any_penalty) {
            PenaltyBufs pb{logits, stride, vocab, history};
            penalty_hash_kernel<<<rows, kPhThreads, 0, stream>>>(a, pb);
            TWD_HIP(hipGetLastError());
        }
        const bool aux = any_short && want_aux(rows, vocab, short_want);
        const SampleStats st{s.wkey, s.wsum, s.wmax, aux ? s.waux : nullptr, __builtin_nanf("")};  // no cap
        WaveStatsBufs wb{logits, stride, vocab, waves, st};
        const dim3 grid((vocab + kWsEntries - 1) / kWsEntries, rows);
        if (aux)
            wave_stats_kernel<1, true><<<grid, kWsThreads, 0, stream>>>(wb);
        else
            wave_stats_kernel<1, false><<<grid, kWsThreads, 0, stream>>>(wb);
        TWD_HIP(hipGetLastError());
        SampleMergeBufs mb{};
        mb.logits = logits;
        mb.stride = stride;
        mb.vocab = vocab;
        mb.waves = waves;
        mb.st = st;
        mb.tokens = tokens;
        if (any_short) {
            merge_kernel<kSampleWaveShift>(waves)<<<rows, kSmThreads, sizeof(SampleMergeShared), stream>>>(a, mb);
            TWD_HIP(hipGetLastError());
        }
        return launch_long(s.lng, st, waves, kSampleWaveRows, logits, stride, vocab, rows, params, tokens, stream);
    }
    SelectBufs b{};
    b.logits = logits;
    b.vocab = vocab;
    b.stride = stride;
    b.history = history;
    b.tokens = tokens;
    b.part_max = s.part_max;
    b.part_sum = s.part_sum;
    b.part_flag = s.part_flag;
    b.part_count = s.part_count;
    b.part_key = s.part_key;
    b.cand = s.cand;
    // every row greedy: the slice blocks finish the rows (one launch instead of two)
    if (!penalty_only && !any_sampled && parts > 1 && s.gbest && s.gctr && s.epoch) {
        *s.epoch = epoch_after(*s.epoch);  // 1 .. 2^31 - 1, never 0
        a.one_pass = 1;
        a.epoch = *s.epoch;
        a.next_epoch = epoch_after(*s.epoch);
        b.gbest = s.gbest;
        b.gctr = s.gctr;
    }
    select_slice_kernel<<<dim3(parts, rows), kSliceThreads, sizeof(SliceShared), stream>>>(a, b);
    TWD_HIP(hipGetLastError());
    if (parts > 1 && !penalty_only && !a.one_pass) {
        select_merge_kernel<<<rows, kMergeThreads, sizeof(MergeShared), stream>>>(a, b);
        TWD_HIP(hipGetLastError());
    }
    if (any_long) {  // their wave records from the penalised logits, then the long path
        const SampleStats st{s.wkey, s.wsum, s.wmax, nullptr, __builtin_nanf("")};  // no merge reads words
        WaveStatsBufs wb{logits, stride, vocab, waves, st};
        wave_stats_kernel<1, false><<<dim3((vocab + kWsEntries - 1) / kWsEntries, rows), kWsThreads, 0, stream>>>(wb);
        TWD_HIP(hipGetLastError());
        return launch_long(s.lng, st, waves, kSampleWaveRows, logits, stride, vocab, rows, params, tokens, stream);
    }
    return TWD_OK;
}

int launch_sample_merge(const SampleStats& st, uint32_t waves, uint32_t rec_rows, const float* logits, uint32_t vocab,
                        uint32_t rows, const twd_row_params* params, uint32_t* tokens, uint32_t* mirror,
                        LongScratch* lng, hipStream_t stream) {
    if (waves == 0 || waves > kSampleMaxWaves) return fail(TWD_E_INVALID, "sample merge: head waves out of range");
    if (rows == 0 || rows > TWD_MAX_ROWS) return fail(TWD_E_INVALID, "sample merge: rows out of range");
    int rc = enable_select_kernels();
    if (rc) return rc;
    SelectArgs a{};
    a.rows = rows;
    a.parts = waves;
    for (uint32_t r = 0; r < rows; ++r) a.p[r] = params[r];
    SampleMergeBufs b{};
    b.logits = logits;
    b.stride = vocab;
    b.vocab = vocab;
    b.waves = waves;
    b.st = st;
    b.tokens = tokens;
    b.mirror = mirror;
    const MergeKernel merge = rec_rows == 16   ? merge_kernel<4>(waves)
                              : rec_rows == 32 ? merge_kernel<5>(waves)
                              : rec_rows == 64 ? merge_kernel<6>(waves)
                                               : nullptr;
    if (!merge) return fail(TWD_E_INVALID, "sample merge: record rows out of range");
    merge<<<rows, kSmThreads, sizeof(SampleMergeShared), stream>>>(a, b);
    TWD_HIP(hipGetLastError());
    return launch_long(lng, st, waves, rec_rows, logits, vocab, vocab, rows, params, tokens, stream);
}

int launch_verify_compare(const uint32_t* row_tokens, uint32_t rows, const uint32_t* drafts,
                          uint32_t n_drafts, twd_verify_result* result, hipStream_t stream) {
    verify_compare_kernel<<<1, 64, 0, stream>>>(row_tokens, rows, drafts, n_drafts, result);
    TWD_HIP(hipGetLastError());
    return TWD_OK;
}

}  // namespace twd

using namespace twd;

extern "C" {

TWD_API int twd_selector_create(uint32_t max_vocab, uint32_t max_rows, twd_selector** out) {
    clear_error();
    if (!out) return fail(TWD_E_INVALID, "null out");
    *out = nullptr;
    if (max_vocab == 0 || max_rows == 0 || max_rows > TWD_MAX_ROWS + 1)
        return fail(TWD_E_INVALID, "max_vocab must be > 0 and max_rows in 1..65");
    if (parts_for(max_vocab) > kMaxParts) return fail(TWD_E_UNSUPPORTED, "max_vocab above 524288");
    int rc0 = enable_select_kernels();
    if (rc0) return rc0;
    twd_selector* s = new twd_selector();
    s->max_vocab = max_vocab;
    const int rc = scratch_alloc(&s->scratch, max_vocab, max_rows);
    if (rc) {
        delete s;
        return rc;
    }
    *out = s;
    return TWD_OK;
}

TWD_API void twd_selector_destroy(twd_selector* s) {
    if (!s) return;
    order_release(s->order);
    draft_side_free(&s->draft);  // waits for the side stream's work
    scratch_free(&s->scratch);
    draft_scratch_free(&s->draft);
    delete s;
}

TWD_API int twd_select(twd_selector* sel, float* logits, uint32_t vocab, uint32_t rows,
                       uint64_t row_stride, const twd_row_params* params,
                       const uint32_t* history, uint32_t* tokens, void* stream) {
    clear_error();
    if (!sel) return fail(TWD_E_INVALID, "null selector");
    if (vocab > sel->max_vocab) return fail(TWD_E_INVALID, "vocab larger than this selector's max_vocab");
    const hipStream_t s = static_cast<hipStream_t>(stream);
    int rc = order_before(sel->order, s);
    if (rc) return rc;
    rc = launch_select(sel->scratch, logits, vocab, rows, row_stride, params, history, tokens, s);
    const int rc2 = order_after(sel->order, s);
    return rc ? rc : rc2;
}

TWD_API int twd_select_noalloc(float* logits, uint32_t vocab, uint32_t rows, uint64_t row_stride,
                               const twd_row_params* params, const uint32_t* history,
                               uint32_t* tokens, void* stream) {
    clear_error();
    if (vocab > kStaticVocab)
        return fail(TWD_E_INVALID, "twd_select_noalloc: vocab above its fixed scratch's 262144 entries");
    if (rows > kStaticRows) return fail(TWD_E_INVALID, "twd_select_noalloc: rows above 64");
    int rc = enable_select_kernels();
    if (rc) return rc;
    SelectScratch s{};
    if ((rc = static_scratch(&s))) return rc;
    return launch_select(s, logits, vocab, rows, row_stride, params, history, tokens,
                         static_cast<hipStream_t>(stream));
}

TWD_API int twd_verify(twd_selector* sel, const float* logits, uint32_t vocab, uint32_t rows,
                       uint64_t row_stride, const twd_row_params* params, uint64_t base_seed,
                       const uint32_t* drafts, uint32_t n_drafts, twd_verify_result* result,
                       void* stream) {
    clear_error();
    if (!sel || !params || !result) return fail(TWD_E_INVALID, "null selector, params or result");
    if (n_drafts > 0 && !drafts) return fail(TWD_E_INVALID, "null drafts");
    if (n_drafts > TWD_MAX_ROWS) return fail(TWD_E_INVALID, "n_drafts must be <= 64");
    if (rows > sel->scratch.max_rows) return fail(TWD_E_INVALID, "rows out of range for this selector");
    const hipStream_t s = static_cast<hipStream_t>(stream);
    int rc = order_before(sel->order, s);
    if (rc) return rc;
    rc = verify_launches(sel, logits, vocab, rows, row_stride, params, base_seed, drafts, n_drafts,
                         result, s);
    const int rc2 = order_after(sel->order, s);
    return rc ? rc : rc2;
}

}  // extern "C"

namespace twd {

int verify_launches(twd_selector* sel, const float* logits, uint32_t vocab, uint32_t rows,
                    uint64_t row_stride, const twd_row_params* params, uint64_t base_seed,
                    const uint32_t* drafts, uint32_t n_drafts, twd_verify_result* result,
                    hipStream_t s) {
    if (n_drafts == 0 || rows == 0)
        return launch_verify_compare(sel->scratch.verify_tokens, 0, drafts, n_drafts, result, s);
    // Only rows 0..min(n_drafts, rows) can be consulted; sample them all, as the reference
    // would on the path it takes.
    const uint32_t k = std::min(n_drafts, rows);
    const uint32_t used = (rows > k) ? k + 1 : k;
    twd_row_params rp[TWD_MAX_ROWS + 1];
    for (uint32_t i = 0; i < used; ++i) {
        rp[i] = *params;
        rp[i].repetition_penalty = 1.0f;
        rp[i].history_len = 0;
        rp[i].uniform = twd_uniform_from_seed(twd_splitmix64(base_seed + i));
    }
    // The selector only reads the rows (penalty is off), so the const cast does not write.
    int rc = launch_select(sel->scratch, const_cast<float*>(logits), vocab, used, row_stride, rp,
                           nullptr, sel->scratch.verify_tokens, s);
    if (rc) return rc;
    return launch_verify_compare(sel->scratch.verify_tokens, used, drafts, n_drafts, result, s);
}

}  // namespace twd
