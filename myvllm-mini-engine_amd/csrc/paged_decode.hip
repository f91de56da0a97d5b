// GQA paged decode attention for gfx950: launch plan, split-K merge and
// the C entry points.  The attention kernel and its design notes are in
// paged_decode_kernel.h.
#include <algorithm>
#include <mutex>

#include "paged_decode_kernel.h"

namespace mvme {
namespace {

// Split-K combine: out = sum_p acc_p 2^(m_p - M) / sum_p l_p 2^(m_p - M).
// Partitions that never saw a valid token carry m = -inf and contribute 0;
// an all-empty sequence produces 0.
// One work-group of whole waves per (sequence, query head), D rounded up to
// 64 threads; thread t < D owns output dim t.  Threads past D take part in
// the partition-maximum and weight loops and feed the identities (-inf for
// the maximum, 0 for the sums) into the reductions, so a wave never reads a
// lane that does not exist.  Every step loads many partitions at once: the
// partition maxima one per thread, then (per window of partitions) the
// weights 2^(m_p - ref) into LDS and each dim's partials eight at a time.
constexpr int kMergeWindow = 2048;  // partition weights held in LDS at once

template <int D>
constexpr int merge_threads() { return (D + kWave - 1) / kWave * kWave; }

// Merge of at most N partitions: every thread loads its dim's partials and all
// (max, sum) pairs at once, without knowing yet how many partitions the
// sequence has (rows past them hold nothing and are dropped), so the launch
// is one memory round trip and no barrier (8 sequences of 512, bf16: the two
// launches 9.4 -> 9.0 us, together with the attention kernel's early page
// lookup).
template <typename T, int D, int N>
__device__ inline void merge_direct(const DecodeArgs& a, int64_t bh, int b) {
    const int tid = threadIdx.x;
    if (tid >= D) return;
    const float* ml = a.ws_ml + bh * a.max_parts * 2;
    const float* acc = a.ws_acc + bh * a.max_parts * D + tid;
    float m[N], l[N], v[N];
#pragma unroll
    for (int p = 0; p < N; ++p) {
        const int row = min(p, a.max_parts - 1);
        m[p] = ml[2 * row];
        l[p] = ml[2 * row + 1];
        v[p] = acc[(int64_t)row * D];
    }
    const int len = seq_tokens(a.lens[b], a.capacity);
    const int nparts = len > 0 ? (len + a.partition - 1) / a.partition : 1;
    if (nparts == 1) return;  // written directly by the attention kernel
    float mx = kNegInf;
#pragma unroll
    for (int p = 0; p < N; ++p) {
        if (p >= nparts) m[p] = kNegInf;
        mx = fmaxf(mx, m[p]);
    }
    const float ref = mx == kNegInf ? 0.f : mx;
    float o = 0.f, sum = 0.f;
#pragma unroll
    for (int p = 0; p < N; ++p) {
        const float w = fast_exp2(m[p] - ref);
        sum += p < nparts ? l[p] * w : 0.f;
        o += p < nparts ? v[p] * w : 0.f;
    }
    static_cast<uint16_t*>(a.out)[bh * D + tid] = T::from_float(sum > 0.f ? o / sum : 0.f);
}

template <typename T, int D>
__global__ __launch_bounds__(256) void paged_decode_merge_kernel(DecodeArgs a) {
    static_assert(D <= 256, "one thread per output dim");
    constexpr int kThreads = merge_threads<D>();
    __shared__ float sm_red[kThreads / kWave];
    __shared__ float sm_w[kMergeWindow];
    const int64_t bh = blockIdx.x;
    const int b = (int)(bh / a.q_heads);
    if (a.max_parts <= 4) {
        merge_direct<T, D, 4>(a, bh, b);
        return;
    }
    if (a.max_parts <= 8) {
        merge_direct<T, D, 8>(a, bh, b);
        return;
    }
    if (a.max_parts <= 16) {
        merge_direct<T, D, 16>(a, bh, b);
        return;
    }
    const int len = seq_tokens(a.lens[b], a.capacity);
    const int nparts = len > 0 ? (len + a.partition - 1) / a.partition : 1;
    if (nparts == 1) return;  // written directly by the attention kernel
    const float* ml = a.ws_ml + bh * a.max_parts * 2;
    const float* acc = a.ws_acc + bh * a.max_parts * D;
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1), wave = tid / kWave;
    constexpr int kWaves = kThreads / kWave;
    const bool owns_dim = tid < D;
    auto block_reduce = [&](float v, bool is_max) __attribute__((always_inline)) {
#pragma unroll
        for (int off = kWave / 2; off > 0; off >>= 1) {
            const float o = __shfl_xor(v, off);
            v = is_max ? fmaxf(v, o) : v + o;
        }
        __syncthreads();  // earlier reads of sm_red are done
        if (lane == 0) sm_red[wave] = v;
        __syncthreads();
        v = sm_red[0];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) v = is_max ? fmaxf(v, sm_red[w]) : v + sm_red[w];
        return v;
    };
    float mx = kNegInf;
    for (int p = tid; p < nparts; p += kThreads) mx = fmaxf(mx, ml[2 * p]);
    mx = block_reduce(mx, true);
    const float ref = mx == kNegInf ? 0.f : mx;
    constexpr int kBatch = 8;
    float o = 0.f, sum = 0.f;
    for (int w0 = 0; w0 < nparts; w0 += kMergeWindow) {
        const int n = min(kMergeWindow, nparts - w0);
        __syncthreads();  // the previous window's weights are no longer read
        for (int p = tid; p < n; p += kThreads) {
            const float w = fast_exp2(ml[2 * (w0 + p)] - ref);
            sm_w[p] = w;
            sum += ml[2 * (w0 + p) + 1] * w;
        }
        __syncthreads();
        if (!owns_dim) continue;
        const float* accw = acc + (int64_t)w0 * D + tid;
        for (int p0 = 0; p0 < n; p0 += kBatch) {
            // Indices past the window's last partition re-read it; the
            // select drops them.
            float av[kBatch], wv[kBatch];
#pragma unroll
            for (int k = 0; k < kBatch; ++k) {
                const int pk = min(p0 + k, n - 1);
                av[k] = accw[(int64_t)pk * D];
                wv[k] = sm_w[pk];
            }
#pragma unroll
            for (int k = 0; k < kBatch; ++k) o += p0 + k < n ? av[k] * wv[k] : 0.f;
        }
    }
    sum = block_reduce(sum, false);
    if (owns_dim) static_cast<uint16_t*>(a.out)[bh * D + tid] = T::from_float(sum > 0.f ? o / sum : 0.f);
}

// Merge of the balanced walk: work-group l merges the unit its share's
// descriptor names (one that began in an earlier share and ends in this
// one).  The unit's pieces are the shares from p0, the one holding its first
// chunk, up to l; share p0 wrote its piece in row slot `slot0` (1 when the
// unit was its last segment), every later one as its first segment (slot 0).
// Shares left empty (fewer chunks than work-groups) wrote nothing: they get
// weight 0 and read the merging share's own row instead, so every load is
// unconditional.  A unit has at most one piece per work-group of the walk:
// thread t reads piece t's (reference, sum) pairs, the block maximum gives
// the reference, and the weights and row offsets go to LDS; each output dim
// then sums its pieces in order, kBatch loads at a time (the same sums, in
// the same order, as one piece after the other; a zero weight adds nothing).
// Work-group g merges share (g mod 8) * kFlatGroups/8 + g/8, the share the
// attention kernel's work-group g computed, so the merge runs on the XCD
// whose L2 holds that share's partials.  Measured against the first version
// (one piece after the other, each a dependent load, and the walk's prefix
// sums recomputed before the first load; µs per call): one sequence of
// 32768 keys 32.0 -> 29.7, two of 8192 27.5 -> 18.3, 8 of 512 11.9 -> 9.6.
template <typename T, int D, int G>
__global__ __launch_bounds__(kLptMax) void paged_decode_flat_merge_kernel(DecodeArgs a) {
    __shared__ float sm_red[G][kLptMax / kWave];
    __shared__ float sm_w[G][kLptMax];
    __shared__ float sm_lw[G][kLptMax];
    __shared__ int64_t sm_row[kLptMax];
    const int64_t l = (blockIdx.x & 7) * (kFlatGroups >> 3) + (blockIdx.x >> 3);
    const FlatMergeDesc dsc = a.ws_flat[l];
    if (dsc.b < 0) return;
    const int64_t total = dsc.total;
    const int64_t p0 = dsc.p0;
    const int n = (int)(l - p0 + 1);
    const int kvh = dsc.r / a.gtiles;
    const int tile0 = (dsc.r - kvh * a.gtiles) * a.tile_heads;
    const int h0 = kvh * a.group + tile0;
    const int heads = matrix_tile<D, G>() ? min(a.tile_heads, a.group - tile0) : G;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const int64_t p = p0 + tid;
    const bool live = tid < n && flat_share_start(p, total) < flat_share_start(p + 1, total);
    const int64_t row = (p * 2 + (tid == 0 ? dsc.slot0 : 0)) * G;
    float m[G], lsum[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        m[g] = live && g < heads ? a.ws_ml[(row + g) * 2] : kNegInf;
        lsum[g] = live && g < heads ? a.ws_ml[(row + g) * 2 + 1] : 0.f;
        float v = m[g];
#pragma unroll
        for (int off = kWave / 2; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
        if (lane == 0) sm_red[g][wave] = v;
    }
    // Empty pieces read the merging share's own row (always written) and
    // are dropped by their zero weight.
    if (tid < n) sm_row[tid] = live ? row : (l * 2) * G;
    __syncthreads();
#pragma unroll
    for (int g = 0; g < G; ++g) {
        float mx = sm_red[g][0];
#pragma unroll
        for (int w = 1; w < kLptMax / kWave; ++w) mx = fmaxf(mx, sm_red[g][w]);
        const float ref = mx == kNegInf ? 0.f : mx;
        const float w = live ? fast_exp2(m[g] - ref) : 0.f;
        if (tid < n) {
            sm_w[g][tid] = w;
            sm_lw[g][tid] = live ? lsum[g] * w : 0.f;
        }
    }
    __syncthreads();
    // Four output dims per thread; when that leaves threads over, kGroups of
    // them share the pieces and meet in LDS.
    constexpr int kVecs = G * D / 4;
    constexpr int kGroups = kLptMax / kVecs;
    static_assert(kGroups >= 1, "one thread per four output dims");
    constexpr int kBatch = 8;
    const int grp = tid / kVecs, idx = tid - grp * kVecs;
    const int g = idx / (D / 4), d = 4 * (idx - g * (D / 4));
    const bool active = grp < kGroups && g < heads;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    float sum = 0.f;
    if (active) {
        for (int t0 = grp; t0 < n; t0 += kBatch * kGroups) {
            f32x4 av[kBatch];
#pragma unroll
            for (int k = 0; k < kBatch; ++k)
                av[k] = *reinterpret_cast<const f32x4*>(a.ws_acc + (sm_row[min(t0 + k * kGroups, n - 1)] + g) * D + d);
#pragma unroll
            for (int k = 0; k < kBatch; ++k) {
                const int t = min(t0 + k * kGroups, n - 1);
                const bool use = t0 + k * kGroups < n && sm_w[g][t] != 0.f;
                const float w = use ? sm_w[g][t] : 0.f;
                sum += use ? sm_lw[g][t] : 0.f;
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] += use ? av[k][i] * w : 0.f;
            }
        }
    }
    if constexpr (kGroups > 1) {
        __shared__ f32x4 sm_o[kGroups * kVecs];
        __shared__ float sm_sum[kGroups * kVecs];
        if (grp < kGroups) {
            sm_o[tid] = o;
            sm_sum[tid] = sum;
        }
        __syncthreads();
        if (grp > 0 || !active) return;
        for (int q = 1; q < kGroups; ++q) {
            o += sm_o[q * kVecs + idx];
            sum += sm_sum[q * kVecs + idx];
        }
    } else if (!active) {
        return;
    }
    uint16_t* out = static_cast<uint16_t*>(a.out) + ((int64_t)dsc.b * a.q_heads + h0 + g) * D + d;
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] = T::from_float(sum > 0.f ? o[i] / sum : 0.f);
}

// Merge of even parts: one work-group per (sequence, query head).  The
// partition length is recomputed from the lengths as the attention kernel
// did; a sequence's rows lie one slot (a.kv_heads * a.gtiles work-groups of G
// rows) apart.  kThreads / D groups of threads take every kGroups-th
// partition, kBatch at a time with a running reference, and meet in LDS.
template <typename T, int D, int G>
__global__ __launch_bounds__(256) void paged_decode_even_merge_kernel(DecodeArgs a) {
    constexpr int kGroups = 256 / D, kBatch = 8;
    __shared__ float sm[kGroups > 1 ? kGroups : 1][3][D];
    const int b = blockIdx.x / a.q_heads, h = blockIdx.x - b * a.q_heads;
    const EvenParts e = even_parts(a, DecodeShape<D>::kTpi * kSplitWaves);
    const int n = lane_value(e.count, b);
    if (n == 1) return;  // written directly by the attention kernel
    const int slot0 = lane_value(e.incl, b) - n;
    const int kvh = h / a.group, hg = h - kvh * a.group;
    const int tile = hg / a.tile_heads;
    const int cols = a.kv_heads * a.gtiles;
    const int64_t row0 = ((int64_t)slot0 * cols + kvh * a.gtiles + tile) * G + (hg - tile * a.tile_heads);
    const int64_t stride = (int64_t)cols * G;
    const int grp = threadIdx.x / D, d = threadIdx.x - grp * D;
    float mx = kNegInf, sum = 0.f, o = 0.f;
    if (grp < kGroups) {
        for (int p0 = grp; p0 < n; p0 += kBatch * kGroups) {
            float m[kBatch], l[kBatch], v[kBatch];
#pragma unroll
            for (int k = 0; k < kBatch; ++k) {
                const int64_t row = row0 + min(p0 + k * kGroups, n - 1) * stride;
                m[k] = a.ws_ml[2 * row];
                l[k] = a.ws_ml[2 * row + 1];
                v[k] = a.ws_acc[row * D + d];
            }
            float bm = mx;
#pragma unroll
            for (int k = 0; k < kBatch; ++k) {
                if (p0 + k * kGroups >= n) m[k] = kNegInf;
                bm = fmaxf(bm, m[k]);
            }
            const float ref = bm == kNegInf ? 0.f : bm;
            const float old = fast_exp2(mx - ref);
            sum *= old;
            o *= old;
            mx = bm;
#pragma unroll
            for (int k = 0; k < kBatch; ++k) {
                const float w = p0 + k * kGroups < n ? fast_exp2(m[k] - ref) : 0.f;
                sum += p0 + k * kGroups < n ? l[k] * w : 0.f;
                o += p0 + k * kGroups < n ? v[k] * w : 0.f;
            }
        }
    }
    if constexpr (kGroups > 1) {
        if (grp < kGroups) {
            sm[grp][0][d] = mx;
            sm[grp][1][d] = sum;
            sm[grp][2][d] = o;
        }
        __syncthreads();
        if (grp > 0) return;
        float all = mx;
#pragma unroll
        for (int g = 1; g < kGroups; ++g) all = fmaxf(all, sm[g][0][d]);
        const float ref = all == kNegInf ? 0.f : all;
        const float own = fast_exp2(mx - ref);
        sum *= own;
        o *= own;
#pragma unroll
        for (int g = 1; g < kGroups; ++g) {
            const float w = fast_exp2(sm[g][0][d] - ref);
            sum += sm[g][1][d] * w;
            o += sm[g][2][d] * w;
        }
    } else if (grp > 0) {
        return;
    }
    static_cast<uint16_t*>(a.out)[(int64_t)blockIdx.x * D + d] = T::from_float(sum > 0.f ? o / sum : 0.f);
}

struct DecodePlan {
    int partition;
    int max_parts;
    int gtile;  // G of the kernel instance
    int gtiles; // query-head tiles per kv head
    int tile_heads; // query heads per tile (at most gtile)
    int waves;  // waves per work-group (kSplitWaves or kWholeWaves; kFlatWaves in the walk)
    bool stream;  // non-temporal K/V loads
    int flat_groups;  // > 0: balanced walk with this many work-groups
    int even_slots;   // > 0: even parts, work-groups per column
    int even_min;     // shortest part
};


// Query heads per kv head from which tiles run on the matrix cores (small calls
// apart, see plan_tiles).  A tile of up to 4 heads costs them the same whatever
// the number; with 2 heads the dot-product kernel is ahead at one unit per CU (32
// sequences of 2048, fp16: 44.6 us against 46.3) and make_decode_plan says where it
// is not, with 4 the matrix cores are (48.4 -> 46.3).
constexpr int64_t kMatrixGroup = 3;
constexpr int64_t kStreamBytes = int64_t(64) << 20;  // K+V bytes within capacity above which loads stream

int decode_tile_tokens(int64_t head_dim) {
    switch (head_dim) {
        case 16: return DecodeShape<16>::kTpi;
        case 32: return DecodeShape<32>::kTpi;
        case 64: return DecodeShape<64>::kTpi;
        case 80: return DecodeShape<80>::kTpi;
        case 96: return DecodeShape<96>::kTpi;
        case 128: return DecodeShape<128>::kTpi;
        case 192: return DecodeShape<192>::kTpi;
        case 256: return DecodeShape<256>::kTpi;
        default: return 0;
    }
}

constexpr int64_t kDeviceCUs = 256;  // MI355X compute units

// Smallest tables, in tokens, over which 8-head tiles take even parts.
constexpr int64_t kEvenCapacity = 2048;

// Query-head tiles of a group: on the matrix cores the fewest tiles of at
// most 8 heads, of equal size (a tile reads all K/V rows of its kv head, so
// one tile of 7 beats seven of 1, and 9 heads are 5 + 4); otherwise tiles that
// divide the group.
// Small calls take the latter too: a wide tile rotates, merges and stores all
// of its heads in one work-group, 1 to 3 us that nothing overlaps, while the
// many narrow ones' repeated reads come from L2.  The lines are in tokens that
// all narrow tiles together may read, each at half a page below the tables'
// capacity.  us per call, wide / narrow, bf16:
// * tiles of 1 or 2 heads: 9/1 heads, 3 x 38 step 8.1 / 5.0; 28/4, 8 x 496 8.0 /
//   6.0; 7/1, 1 x 3440 (24 k tokens; 2 of them 48 k) 12.0 / 11.5 (12.7 / 13.2); 5/1,
//   16 x 608 (48 k) 8.2 / 9.7; 5/1 of 64, 40 x 304 (61 k) 7.1 / 7.2; 6/1, 96 x 128
//   (74 k) 7.3 / 8.5;
// * three heads, which one tile of 4 holds: 8 x 32 step 5.9 / 4.9; 16 x 576 (26 k)
//   8.2 / 8.5; 19 x 832 (47 k) 8.5 / 10.8; 6 x 3072 (53 k) 8.3 / 11.2;
// * tiles of 4: 12/4, 24 x 144 step 9.9 / 7.6; 8/1, 2 x 1536 11.9 / 11.2; 48/8, 4 x
//   592 9.9 / 9.2; over tables that take even parts 8/1, 2 x 4096 (16 k) 12.3 / 15.0,
//   12/1, 3 x 4624 (42 k) 12.2 / 15.4; and more of them than CUs, 64/4, 18 x 141
//   7.6 / 8.9;
// * groups of 4, 8, ... in tiles of 2 (tiles of 4 / of 2): 12/1, 39 x 24 step (5 k)
//   9.4 / 6.6, 8/1, 18 x 168 step (12 k) 10.8 / 7.6, both on odd pages; 12/1, 72 x 48
//   (17 k) 4.7 / 4.9; 8/4, 4 x 512 (25 k) 7.0 / 7.9.
constexpr int64_t kNarrowTokens = 48 << 10, kNarrowThree = 28 << 10, kPairTokens = 20 << 10;
void plan_tiles(DecodePlan& p, int64_t group, int64_t head_dim, int64_t kv_units, int64_t cap, int64_t block_size) {
    const bool matrix = head_dim == 64 || head_dim == 128;
    const double tokens = (double)kv_units * (double)(cap - block_size / 2);
    const bool fours = group % 4 == 0 && !(matrix && tokens * (double)(group / 2) <= (double)kPairTokens);
    const int64_t narrow = fours ? 4 : group % 2 == 0 ? 2 : 1;
    bool small = tokens * (double)(group / narrow) <= (double)(group == 3 ? kNarrowThree : kNarrowTokens);
    if (fours) small = small && kv_units * (group / 4) <= kDeviceCUs && (head_dim != 128 || cap < kEvenCapacity);
    if (matrix && group >= kMatrixGroup && !small) {
        const int64_t tiles = (group + 7) / 8;
        const int64_t heads = (group + tiles - 1) / tiles;
        p.gtiles = (int)((group + heads - 1) / heads);
        p.tile_heads = (int)heads;
        p.gtile = heads <= 4 ? 4 : 8;
        return;
    }
    p.gtile = (int)narrow;
    p.gtiles = (int)(group / narrow);
    p.tile_heads = p.gtile;
}

// Smallest K+V capacity of a 128-dim unit from which the balanced walk takes a plan of
// `units` units, in bytes; 0: none.  us per call, other plan -> walk (16/8
// heads, bf16, pages of 16; first ragged U[1,ctx], then all ctx):
// * fewer units than CUs (split-K): 2048 tokens (1 MiB) 24 sequences 23.0 ->
//   28.0, 39.2 -> 39.6; 2600 tokens 24.4 -> 23.7, 34.6 -> 32.9 (16 sequences),
//   32.2 -> 28.5, 49.6 -> 46.1 (24); 4000 tokens 50.2 -> 39.9, 70.3 -> 67.4.
// * one unit per CU: 1400 tokens, 32 sequences 23.7 -> 24.3, 32.0 -> 33.2; 2048
//   tokens 34.9 -> 30.2, 46.3 -> 45.2; 4000 tokens 60.0 -> 52.3.
// * up to 1.25 per CU, some CUs with two units and others with one: 34
//   sequences of 1000 25.2 -> 22.3, 35.7 -> 29.3, of 4000 81.1 -> 55.0, 131.4 ->
//   90.9; 40 of 1000 25.1 -> 25.5, 38.6 -> 33.6.
// * up to 1.5: 48 of 1000 25.8 -> 27.8, 41.3 -> 39.2; of 2000 44.5 -> 42.9, 76.1
//   -> 66.6.
// * up to 1.9: 56 of 2000 46.8 -> 48.2, 81.3 -> 77.5; of 4000 86.3 -> 82.4,
//   157.0 -> 146.7; two per CU (64 of 4000) 90.8 -> 92.3: none.
// The walk's pieces of 8-head tiles end more slowly: up to one unit per CU 62
// sequences of 3000 (28/4 heads) 53.8 -> 51.8, 64 of 2048 (32/4) 40.5 -> 50.2;
// above, 48 of 4000 (40/8) 84.3 -> 81.9, 40 of 2000 38.7 -> 47.0.
int64_t walk_unit_bytes(int64_t units, int gtile) {
    const int64_t mib = int64_t(1) << 20;
    const bool one_per_cu = units >= kDeviceCUs - kDeviceCUs / 16 && units <= kDeviceCUs;
    if (gtile == 8) return one_per_cu ? mib * 3 / 2 : units <= kDeviceCUs * 3 / 2 ? 2 * mib : 0;
    if (units < kDeviceCUs * 3 / 8) return 2 * mib;
    if (units <= kDeviceCUs) return mib * 5 / 4;
    if (units <= kDeviceCUs * 5 / 4) return mib / 2;
    if (units <= kDeviceCUs * 3 / 2) return mib;
    return units <= kDeviceCUs * 15 / 8 ? mib * 3 / 2 : 0;
}

// Partition length of a split over tiles of 1 to 4 heads of 128: the number of
// partitions n that minimises the iterations the busiest CU runs, half at full
// tables and half at tables filled a little over half (ragged batches), plus
// a share per partition for its start, its end and the merge.  A target of two
// work-groups per CU alone leaves some CUs with three and others with two: 24
// sequences of 2048, 8 kv heads (192 units): 3 partitions 42.9 us (26.7 for
// U[1,2048]), 4 partitions -- three per CU -- 36.5 (22.1).
// (8/8 heads: 42.8 -> 37.9 and 26.2 -> 21.3.)
int64_t split_partition(int64_t cap, int64_t units, int64_t step) {
    const int64_t steps = (cap + step - 1) / step;
    int64_t best = 1;
    double best_cost = 1e300;
    for (int64_t n = 2; n <= 32 && n <= steps; ++n) {
        const int64_t iterations = (steps + n - 1) / n;
        const double groups = (double)(units * n);
        const double full = (double)((units * n + kDeviceCUs - 1) / kDeviceCUs);
        const double ragged = std::max(1.0, 0.55 * groups / (double)kDeviceCUs);
        const double cost = 0.5 * (full + ragged) * (double)iterations + 0.15 * (double)n;
        if (cost < best_cost) best_cost = cost, best = n;
    }
    return (steps + best - 1) / best * step;
}

// Host-side plan (lengths stay on the device, so it depends on the table
// capacity only).  Long units (walk_unit_bytes) take the balanced walk, unless
// `walk` is off, where only units of kLongUnitBytes numbering at most one per
// CU do (what a call without room for the walk's partials had).  Otherwise, enough (sequence, kv
// head) units to occupy every CU, a capacity of one 16-wave step, or two
// steps with more than a quarter of the CUs' worth of units: one work-group
// per unit over the whole context, merged in LDS (8 waves; with two
// work-groups per CU holding every unit, long sequences paired with short
// ones; below two 16-wave steps, 4 waves when the units outnumber the CUs).
// (A "16-wave step" is 16 wave iterations of tokens, the unit the
// thresholds were measured in.)  Otherwise split-K into partitions of 4-wave
// work-groups, sized to give every CU about two work-groups (at least one
// 4-wave step each), plus a merge kernel.  `requested` > 0 forces split-K
// with that partition length (rounded to the wave tiling), -1 the balanced
// walk (batch <= 256).
//
// Measured at head_dim 128 (bf16, block 16, 16/8 heads, µs per call in a
// graph): whole-sequence against split-K at 64/128/256 keys.
// * ctx 128: whole 4.9-5.1, any split about 2 µs more (the merge launch).
// * ctx 256: level up to 64 units; whole ahead from 128 units.
// * ctx 512: split at 64 ahead up to 64 units (1 unit 7.96 -> 6.87, 64 units
//   8.18 -> 7.82); whole ahead from 128 units (128 units 9.01 vs 9.98).
// (All of these on the dot-product loop.  Splits of pairs and of wider groups at 64
// and 128 dims have since run the matrix cores' loop, with the same lines.)
// * ctx 1024-4096 with 8-64 units: the best partition gives about 512
//   work-groups (1024 keys x 8 units: 256-key parts 9.69, 64-key 7.30; 1024
//   x 64: 11.61 -> 9.93 at 128; 2048 x 32: 11.56 -> 10.48 at 128); the
//   earlier plan took at least 256 keys for a target of 1024 work-groups.
DecodePlan make_decode_plan(int64_t batch, int64_t q_heads, int64_t kv_heads, int64_t head_dim,
                            int64_t block_size, int64_t table_width, int64_t requested, bool walk = true) {
    DecodePlan p{};
    const int64_t group = q_heads / kv_heads;
    const int64_t cap = table_width * block_size;
    plan_tiles(p, group, head_dim, batch * kv_heads, cap, block_size);
    const int64_t tile = decode_tile_tokens(head_dim);
    const int64_t units = batch * kv_heads * p.gtiles;
    const int64_t split_step = tile * kSplitWaves;
    const int64_t whole_step = tile * 16;  // the capacity unit the thresholds below were measured in
    int64_t part;
    const bool whole = units >= kDeviceCUs - kDeviceCUs / 16 || cap <= whole_step ||
                       (cap <= 2 * whole_step && units > kDeviceCUs / 4);
    if (requested <= 0 && whole) {
        // Below two whole steps (512 tokens at D=128): 8 waves (a 128-token
        // context in one iteration of loads) while the units fit the CUs, 4
        // beyond (more work-groups per CU).  µs per call: B1 / ctx 128 fp16 4.85 -> 4.77,
        // B4 / ctx 256 6.82 -> 6.00, B32 / ctx 256 bf16 8.76 -> 7.32; but
        // B64 / ctx 128 7.18 -> 7.39 (512 units), hence 4 there.
        const int short_waves = units <= kDeviceCUs ? kWholeWaves : kSplitWaves;
        p.waves = cap < 2 * whole_step ? short_waves : kWholeWaves;
        part = (cap + tile - 1) / tile * tile;
    } else {
        p.waves = kSplitWaves;
        if (requested > 0) {
            part = requested;
        } else if (group <= 4 && head_dim == 128) {
            part = split_partition(cap, units, split_step);
        } else {
            // Wide tiles of 64 dims gain from more and shorter partitions: 14/2 heads, 60 sequences
            // U[1,1300] 22.2 -> 16.5 at 128 keys, 20 of U[1,4000] 22.6 -> 17.6.
            const int64_t target = head_dim == 64 && p.gtile == 8 ? 5 * kDeviceCUs : 2 * kDeviceCUs;
            part = (cap * units + target - 1) / target;
        }
        part = (part + split_step - 1) / split_step * split_step;
        const int64_t cap_steps = (cap + split_step - 1) / split_step * split_step;
        if (part > cap_steps) part = cap_steps;
    }
    p.partition = (int)part;
    p.max_parts = (int)((cap + part - 1) / part);
    // Long units (walk_unit_bytes) or a request (requested == -1) take the
    // balanced walk.  With one work-group per unit the CUs holding the shortest
    // units, or one unit where others hold two, idle while the rest stream
    // alone, whatever the order; split-K partitions sized by capacity leave
    // ragged batches with empty partitions and uneven CUs.  With two units per
    // CU the longest-first order already balances them.
    const int64_t long_bytes = walk && head_dim == 128 ? walk_unit_bytes(units, p.gtile)
                               : units <= kDeviceCUs   ? kLongUnitBytes
                                                       : 0;
    const bool long_units = long_bytes > 0 && (double)cap * (double)head_dim * 4.0 >= (double)long_bytes;
    // Even parts: 8-head tiles over tables of 2048 tokens and more.
    const bool even = requested <= 0 && requested != -1 && !whole && p.gtile == 8 && head_dim == 128 && batch <= kWave &&
                      cap >= kEvenCapacity;
    if (even) {
        p.even_slots = (int)(kEvenGroups / (kv_heads * p.gtiles));
        p.even_min = (int)(4 * split_step);
        p.max_parts = 1;
    }
    const bool flat = !even && batch <= kLptMax &&
                      (requested == -1 || (requested <= 0 && long_units));
    if (flat) {
        p.flat_groups = kFlatGroups;
        p.waves = kFlatWaves;
        p.max_parts = 1;
    }
    // Pairs of heads on the matrix cores, whose loop keeps loads in flight but
    // starts and ends more slowly (dot products / matrix cores, us per call,
    // 16/8 heads unless noted).
    // At 128 dims, on pages that hold whole iterations (2/1 heads, 3 x 2928 on
    // pages of 8 10.5 / 12.8; 8/4, 39 x 840 on pages of 24 21.1 / 24.2):
    // * splits of up to 160 units: 8 of 512 step 10.0 / 9.7, 16 of U[1,1024]
    //   13.2 / 12.5; 26 of 720 18.6 / 21.0, 26 of 1088 24.0 / 25.5, 23 of 2816 step
    //   44.8 / 47.1;
    // * two long units on most CUs: 64 of U[1,4096] 95.0 / 92.5, 420 units of
    //   U[1,1792] 41.0 / 38.8; 400 of U[1,928] 23.4 / 25.9, 344 of U[1,2304] 62.0 /
    //   64.8, 376 of 1536 step 53.8 / 56.6, one per CU (32 of 2048) 44.6 / 45.8.
    // At 64 dims where pages hold runs of 16 tokens but not the dot products'
    // iterations of 32, which then look up every token's page: 64 of 1000 39.7 /
    // 29.1, 48 of U[1,2000] 35.2 / 29.3 (pages of 256, 128 of 1024 52.7 / 57.0, of
    // 24, 16 of 700 12.6 / 17.2); but not for many short units: 800 of 96 step 10.6
    // / 11.3, 1376 of 192 18.0 / 21.5, 3312 of 480 step 52.9 / 58.0 (768 of 464 step
    // 24.5 / 22.3, 1552 of 864 step 86.1 / 72.0).
    const bool matrix_pairs =
        head_dim == 128 ? block_size % tile == 0 &&
                              (p.max_parts > 1 ? units <= kDeviceCUs * 5 / 8
                                               : p.waves == kWholeWaves && units >= kDeviceCUs * 3 / 2 &&
                                                     units <= 2 * kDeviceCUs && cap >= 1536)
                        : head_dim == 64 && block_size % 32 == 16 && 2 * units <= 5 * cap;
    if (group == 2 && !flat && matrix_pairs) {
        p.gtile = 4;
        p.tile_heads = 2;
    }
    // In floating point: the size query runs before any shape check, where the
    // integer product could overflow.  The walk's kernels always load with the
    // non-temporal hint.
    p.stream = flat || (double)batch * (double)cap * (double)kv_heads * (double)head_dim * 4.0 > (double)kStreamBytes;
    return p;
}

template <typename T, int D, int G, int NW, bool STREAM>
void launch_decode_kernel_pro(const DecodeArgs& a, dim3 grid, bool page_uniform, hipStream_t s) {
    if constexpr (decode_fused_capable<D>()) {
        if (a.prologue != 0) {
            launch_decode_fused<T, D, G, NW, STREAM>(a, grid, page_uniform, s);
            return;
        }
    }
    launch_decode_kernel<T, D, G, NW, STREAM, false>(a, grid, page_uniform, s);
}

template <typename T, int D, int G, int NW>
void launch_decode_nw(const DecodeArgs& a, int units, bool page_uniform, bool stream, hipStream_t s) {
    const dim3 grid(a.flat_groups > 0  ? a.flat_groups
                    : a.even_slots > 0 ? a.even_slots * a.kv_heads * a.gtiles
                                       : units,
                    a.max_parts);
    if (stream) {
        launch_decode_kernel_pro<T, D, G, NW, true>(a, grid, page_uniform, s);
        return;
    }
    launch_decode_kernel_pro<T, D, G, NW, false>(a, grid, page_uniform, s);
}

template <typename T, int D, int G>
void launch_decode(const DecodeArgs& a, const DecodePlan& p, int units, bool page_uniform, hipStream_t s) {
    if (p.waves == kWholeWaves) launch_decode_nw<T, D, G, kWholeWaves>(a, units, page_uniform, p.stream, s);
    else launch_decode_nw<T, D, G, kSplitWaves>(a, units, page_uniform, p.stream, s);
    if constexpr (even_tile<D, G>()) {
        if (a.even_slots > 0) {
            hipLaunchKernelGGL((paged_decode_even_merge_kernel<T, D, G>), dim3(a.batch * a.q_heads), dim3(256), 0, s, a);
            return;
        }
    }
    if (a.flat_groups > 0)
        hipLaunchKernelGGL((paged_decode_flat_merge_kernel<T, D, G>), dim3(a.flat_groups), dim3(kLptMax), 0, s, a);
    else if (a.max_parts > 1)
        hipLaunchKernelGGL((paged_decode_merge_kernel<T, D>), dim3(a.batch * a.q_heads),
                           dim3(merge_threads<D>()), 0, s, a);
}

template <typename T, int D>
void launch_decode_g(const DecodeArgs& a, const DecodePlan& p, int units, bool page_uniform, hipStream_t s) {
    if constexpr (max_gtile<D>() >= 8) {
        if (p.gtile == 8) {
            launch_decode<T, D, 8>(a, p, units, page_uniform, s);
            return;
        }
    }
    if (p.gtile == 4) launch_decode<T, D, 4>(a, p, units, page_uniform, s);
    else if (p.gtile == 2) launch_decode<T, D, 2>(a, p, units, page_uniform, s);
    else launch_decode<T, D, 1>(a, p, units, page_uniform, s);
}

template <typename T>
void launch_decode_d(const DecodeArgs& a, int64_t head_dim, const DecodePlan& p, int units, bool pu,
                     hipStream_t s) {
    switch (head_dim) {
        case 16: launch_decode_g<T, 16>(a, p, units, pu, s); break;
        case 32: launch_decode_g<T, 32>(a, p, units, pu, s); break;
        case 64: launch_decode_g<T, 64>(a, p, units, pu, s); break;
        case 80: launch_decode_g<T, 80>(a, p, units, pu, s); break;
        case 96: launch_decode_g<T, 96>(a, p, units, pu, s); break;
        case 128: launch_decode_g<T, 128>(a, p, units, pu, s); break;
        case 192: launch_decode_g<T, 192>(a, p, units, pu, s); break;
        case 256: launch_decode_g<T, 256>(a, p, units, pu, s); break;
    }
}

constexpr int64_t kMaxCapacity = 1048576;     // tokens a block table may address
constexpr int64_t kMaxBatchHeads = 2147483647; // batch * q_heads

int check_decode_shapes(int64_t batch, int64_t q_heads, int64_t kv_heads, int64_t head_dim,
                        int64_t num_blocks, int64_t block_size, int64_t table_width, int dtype) {
    if (!valid_dtype(dtype)) return fail(MVME_EINVAL, "FP16/BF16 required");
    if (batch <= 0 || q_heads <= 0 || kv_heads <= 0 || num_blocks <= 0)
        return fail(MVME_EINVAL, "empty batch/heads/cache");
    if (block_size <= 0) return fail(MVME_EINVAL, "block size mismatch");
    if (q_heads % kv_heads != 0) return fail(MVME_EINVAL, "head dimension or GQA mismatch");
    if (decode_tile_tokens(head_dim) == 0)
        return fail(MVME_EINVAL, "supported head_dim: 16,32,64,80,96,128,192,256");
    if (table_width <= 0) return fail(MVME_EINVAL, "invalid block table");
    if (block_size > kMaxCapacity || table_width > kMaxCapacity || table_width * block_size > kMaxCapacity)
        return fail(MVME_EINVAL, "maximum table capacity is 1M tokens");
    if (batch > kMaxBatchHeads || q_heads > kMaxBatchHeads || batch * q_heads > kMaxBatchHeads)
        return fail(MVME_EINVAL, "batch/head product too large");
    return MVME_OK;
}

}  // namespace
}  // namespace mvme

using namespace mvme;

namespace mvme {
namespace {

size_t decode_workspace(int64_t batch, int64_t q_heads, int64_t kv_heads, int64_t head_dim, int64_t block_size,
                        int64_t table_width, int64_t partition_tokens, bool walk) {
    if (batch <= 0 || q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads != 0 || block_size <= 0 ||
        table_width <= 0 || decode_tile_tokens(head_dim) == 0)
        return 0;
    // The limits mvme_paged_attention enforces; inside them every product of
    // the plan fits its type.
    if (block_size > kMaxCapacity || table_width > kMaxCapacity || table_width * block_size > kMaxCapacity ||
        batch > kMaxBatchHeads || q_heads > kMaxBatchHeads || batch * q_heads > kMaxBatchHeads)
        return 0;
    const DecodePlan p = make_decode_plan(batch, q_heads, kv_heads, head_dim, block_size, table_width,
                                          partition_tokens, walk);
    if (p.flat_groups > 0)
        return (size_t)p.flat_groups * 2 * p.gtile * (head_dim + 2) * sizeof(float) +
               (size_t)p.flat_groups * sizeof(FlatMergeDesc);
    if (p.even_slots > 0)
        return (size_t)p.even_slots * kv_heads * p.gtiles * p.gtile * (head_dim + 2) * sizeof(float);
    if (p.max_parts <= 1) return 0;
    return (size_t)batch * q_heads * p.max_parts * (head_dim + 2) * sizeof(float);
}

// A caller's workspace too small (or misaligned) for a plan that the walk's
// longer reach gave it: `walk` off, the plan without it, which needs less or
// none.  Returns what the chosen plan needs.
size_t fit_workspace(int64_t batch, int64_t q_heads, int64_t kv_heads, int64_t head_dim, int64_t block_size,
                     int64_t table_width, int64_t partition_tokens, const void* workspace, size_t bytes,
                     bool& walk) {
    walk = true;
    const size_t need = decode_workspace(batch, q_heads, kv_heads, head_dim, block_size, table_width,
                                         partition_tokens, true);
    if (need == 0 || (workspace != nullptr && bytes >= need && (reinterpret_cast<uintptr_t>(workspace) & 15u) == 0))
        return need;
    walk = false;
    return decode_workspace(batch, q_heads, kv_heads, head_dim, block_size, table_width, partition_tokens, false);
}

}  // namespace
}  // namespace mvme

extern "C" size_t mvme_paged_attention_workspace_size(int64_t batch, int64_t q_heads, int64_t kv_heads,
                                                      int64_t head_dim, int64_t block_size,
                                                      int64_t table_width, int64_t partition_tokens) {
    return decode_workspace(batch, q_heads, kv_heads, head_dim, block_size, table_width, partition_tokens, true);
}

namespace mvme {
namespace {

// The fused prologue's inputs (mode 0: none).
struct DecodePrologue {
    int mode;
    const void* new_k;
    const void* new_v;
    int64_t k_stride, v_stride, q_stride;
    const void* q_weight;
    const void* k_weight;
    const void* cos;
    const void* sin;
    void* q_out;
    float eps;
};

// Division of t < 2^31 by a block size b as a product: with s = floor(log2(b - 1))
// and m = ceil(2^(32+s) / b) < 2^32, t * m / 2^(32+s) exceeds t / b by t * e / (b *
// 2^(32+s)) with e = m * b - 2^(32+s) < b <= 2^(s+1), less than 1 / b, so the
// integer part is the quotient.  (b = 1, whose factor would be 2^32, adds t itself.)
void magic_divisor(DecodeArgs& a, int64_t block_size) {
    if (block_size == 1) {
        a.block_one = ~0u;
        return;
    }
    a.block_rest = 63 - __builtin_clzll((unsigned long long)(block_size - 1));
    a.block_magic = (uint32_t)(((1ull << (32 + a.block_rest)) + block_size - 1) / block_size);
}

// Shapes checked, workspace sized: plan the call and launch its kernels.
int launch_paged_attention(void* out, const void* query, const void* key_cache, const void* value_cache,
                           const int64_t* block_tables, const int64_t* context_lens, int64_t batch,
                           int64_t q_heads, int64_t kv_heads, int64_t head_dim, int64_t num_blocks,
                           int64_t block_size, int64_t table_width, int64_t partition_tokens, int dtype,
                           size_t need, bool walk, void* workspace, void* stream,
                           const DecodePrologue* pro = nullptr) {
    const DecodePlan p = make_decode_plan(batch, q_heads, kv_heads, head_dim, block_size, table_width,
                                          partition_tokens, walk);
    const int64_t group = q_heads / kv_heads;
    const int64_t units = batch * kv_heads * p.gtiles;
    if (units > 2147483647) return fail(MVME_EINVAL, "batch/head product too large");
    DecodeArgs a{};
    a.out = out;
    a.query = query;
    a.key_cache = key_cache;
    a.value_cache = value_cache;
    a.tables = block_tables;
    a.lens = context_lens;
    if (need > 0) {
        a.ws_acc = static_cast<float*>(workspace);
        a.ws_ml = a.ws_acc + (p.flat_groups > 0  ? (int64_t)p.flat_groups * 2 * p.gtile
                              : p.even_slots > 0 ? (int64_t)p.even_slots * kv_heads * p.gtiles * p.gtile
                                                 : batch * q_heads * p.max_parts) * head_dim;
        // After the partial rows (a multiple of 16 bytes: 256 shares x 2 x G
        // x (D + 2) floats).
        if (p.flat_groups > 0) {
            if ((reinterpret_cast<uintptr_t>(workspace) & 15u) != 0)
                return fail(MVME_EINVAL, "the balanced walk needs a 16-byte aligned workspace");
            a.ws_flat = reinterpret_cast<FlatMergeDesc*>(a.ws_ml + (int64_t)p.flat_groups * 2 * p.gtile * 2);
        }
    }
    a.q_heads = (int)q_heads;
    a.kv_heads = (int)kv_heads;
    a.group = (int)group;
    a.gtiles = p.gtiles;
    a.tile_heads = p.tile_heads;
    a.num_blocks = num_blocks;
    a.block_size = (int)block_size;
    a.block_shift = (block_size & (block_size - 1)) == 0 ? __builtin_ctzll((unsigned long long)block_size) : -1;
    magic_divisor(a, block_size);
    a.table_width = (int)table_width;
    a.capacity = (int)(table_width * block_size);
    a.partition = p.partition;
    a.max_parts = p.max_parts;
    a.even_slots = p.even_slots;
    a.even_min = p.even_min;
    a.even_few = (int)(kEvenFew / (kv_heads * p.gtiles));
    a.lpt_batch = p.flat_groups == 0 && p.even_slots == 0 && p.max_parts == 1 && batch >= 2 && batch <= kLptMax ? (int)batch : 0;
    // Two 8-wave work-groups per CU hold every unit at once (units in
    // (CUs, 2 CUs]): pair long sequences with short ones.  Longest first
    // alone put the k-th and the (k + batch/2)-th longest on one CU: 64
    // sequences of contexts U[1,2048] (bf16, block 16) 54.8 -> 47.8 µs.
    a.lpt_pair = a.lpt_batch > 0 && p.waves == kWholeWaves && units > kDeviceCUs && units <= 2 * kDeviceCUs;
    a.flat_groups = p.flat_groups;
    a.batch = (int)batch;
    a.scale_log2 = kLog2e / sqrtf((float)head_dim);
    if (pro && pro->mode != 0) {
        a.prologue = pro->mode;
        a.new_k = static_cast<const uint16_t*>(pro->new_k);
        a.new_v = static_cast<const uint16_t*>(pro->new_v);
        a.k_stride = pro->k_stride;
        a.v_stride = pro->v_stride;
        a.q_stride = pro->q_stride;
        a.q_weight = static_cast<const uint16_t*>(pro->q_weight);
        a.k_weight = static_cast<const uint16_t*>(pro->k_weight);
        a.cos = static_cast<const uint16_t*>(pro->cos);
        a.sin = static_cast<const uint16_t*>(pro->sin);
        a.q_out = static_cast<uint16_t*>(pro->q_out);
        a.eps = pro->eps;
    }
    const bool page_uniform = block_size % decode_tile_tokens(head_dim) == 0;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == MVME_FP16) launch_decode_d<Half>(a, head_dim, p, (int)units, page_uniform, s);
    else launch_decode_d<BFloat16>(a, head_dim, p, (int)units, page_uniform, s);
    return check_launch("paged attention");
}

// Split-K scratch of the allocation-free entry point: one array per device,
// held until the process ends.  The kernels write every partial they later
// read, so nothing in it needs clearing between calls.
constexpr size_t kScratchBytes = size_t(8) << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

// Device address of `scratch` on each device, resolved on the first call made
// with that device current (the host-side name is only a handle).
constexpr int kMaxDevices = 64;
std::mutex g_scratch_lock;
void* g_scratch_ptr[kMaxDevices] = {};

int device_scratch(void** ptr) {
    int device = -1;
    if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices)
        return fail(MVME_ELAUNCH, "paged attention (no-alloc): no usable current HIP device");
    std::lock_guard<std::mutex> guard(g_scratch_lock);
    if (g_scratch_ptr[device] == nullptr) {
        void* address = nullptr;
        const hipError_t err = hipGetSymbolAddress(&address, HIP_SYMBOL(scratch));
        if (err != hipSuccess || address == nullptr)
            return fail(MVME_ELAUNCH, std::string("paged attention (no-alloc): scratch address: ") +
                                          hipGetErrorString(err));
        g_scratch_ptr[device] = address;
    }
    *ptr = g_scratch_ptr[device];
    return MVME_OK;
}

}  // namespace
}  // namespace mvme

extern "C" int mvme_paged_attention(void* out, const void* query, const void* key_cache,
                                    const void* value_cache, const int64_t* block_tables,
                                    const int64_t* context_lens, int64_t batch, int64_t q_heads,
                                    int64_t kv_heads, int64_t head_dim, int64_t num_blocks,
                                    int64_t block_size, int64_t table_width, int64_t partition_tokens,
                                    int dtype, void* workspace, size_t workspace_bytes, void* stream) {
    if (int rc = check_decode_shapes(batch, q_heads, kv_heads, head_dim, num_blocks, block_size,
                                     table_width, dtype))
        return rc;
    if (!out || !query || !key_cache || !value_cache || !block_tables || !context_lens)
        return fail(MVME_EINVAL, "paged attention received a null pointer");
    bool walk;
    const size_t need = fit_workspace(batch, q_heads, kv_heads, head_dim, block_size, table_width,
                                      partition_tokens, workspace, workspace_bytes, walk);
    if (need > 0 && (workspace == nullptr || workspace_bytes < need))
        return fail(MVME_EWORKSPACE, "paged attention workspace too small: need " + std::to_string(need) +
                                         " bytes, got " + std::to_string(workspace_bytes));
    return launch_paged_attention(out, query, key_cache, value_cache, block_tables, context_lens, batch,
                                  q_heads, kv_heads, head_dim, num_blocks, block_size, table_width,
                                  partition_tokens, dtype, need, walk, workspace, stream);
}

namespace {
bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
}  // namespace

extern "C" int mvme_paged_attention_decode_write(
    void* out, const void* query, void* key_cache, void* value_cache, const int64_t* block_tables,
    const int64_t* context_lens, int64_t batch, int64_t q_heads, int64_t kv_heads, int64_t head_dim,
    int64_t num_blocks, int64_t block_size, int64_t table_width, int64_t partition_tokens, int dtype,
    const void* new_key, const void* new_value, int64_t key_token_stride, int64_t value_token_stride,
    const void* q_weight, const void* k_weight, const void* cos, const void* sin, float eps,
    int64_t query_token_stride, void* q_out, void* workspace, size_t workspace_bytes, void* stream) {
    if (int rc = check_decode_shapes(batch, q_heads, kv_heads, head_dim, num_blocks, block_size,
                                     table_width, dtype))
        return rc;
    if (!out || !query || !key_cache || !value_cache || !block_tables || !context_lens || !new_key || !new_value)
        return fail(MVME_EINVAL, "paged decode with KV write received a null pointer");
    if (head_dim != 16 && head_dim != 32 && head_dim != 64 && head_dim != 128 && head_dim != 256)
        return fail(MVME_EINVAL, "paged decode with KV write supports head_dim 16,32,64,128,256");
    const bool rope = q_weight != nullptr;
    if (rope && (!k_weight || !cos || !sin))
        return fail(MVME_EINVAL, "paged decode with norm/RoPE needs q_weight, k_weight, cos and sin");
    if (rope && (!(eps > 0.f) || !__builtin_isfinite(eps)))
        return fail(MVME_EINVAL, "eps must be positive, finite and representable in FP32");
    if (key_token_stride < kv_heads * head_dim || value_token_stride < kv_heads * head_dim ||
        (rope && query_token_stride < q_heads * head_dim))
        return fail(MVME_EINVAL, "Q/K/V token stride smaller than a row");
    const bool aligned = aligned16(query) && aligned16(key_cache) && aligned16(value_cache) &&
                         aligned16(new_key) && aligned16(new_value) && key_token_stride % 8 == 0 &&
                         value_token_stride % 8 == 0 &&
                         (!rope || (aligned16(q_weight) && aligned16(k_weight) && aligned16(cos) &&
                                    aligned16(sin) && query_token_stride % 8 == 0 &&
                                    (q_out == nullptr || aligned16(q_out))));
    if (!aligned) return fail(MVME_EINVAL, "paged decode with KV write needs 16-byte aligned rows");
    if (rope && q_out != nullptr) {
        // Every wave (and every split-K partition) reads the raw query rows
        // while the first partition writes the rotated rows to q_out, so the
        // two byte ranges must be disjoint (an in-place rotation belongs to
        // the two-launch sequence).
        const uintptr_t q_lo = reinterpret_cast<uintptr_t>(query);
        const uintptr_t q_hi = q_lo + (uintptr_t)(((batch - 1) * query_token_stride + q_heads * head_dim) * 2);
        const uintptr_t o_lo = reinterpret_cast<uintptr_t>(q_out);
        const uintptr_t o_hi = o_lo + (uintptr_t)(batch * q_heads * head_dim * 2);
        if (o_lo < q_hi && q_lo < o_hi)
            return fail(MVME_EINVAL, "q_out must not overlap the raw query rows");
    }
    bool walk;
    const size_t need = fit_workspace(batch, q_heads, kv_heads, head_dim, block_size, table_width,
                                      partition_tokens, workspace, workspace_bytes, walk);
    if (need > 0 && (workspace == nullptr || workspace_bytes < need))
        return fail(MVME_EWORKSPACE, "paged attention workspace too small: need " + std::to_string(need) +
                                         " bytes, got " + std::to_string(workspace_bytes));
    DecodePrologue pro{};
    pro.mode = rope ? 2 : 1;
    pro.new_k = new_key;
    pro.new_v = new_value;
    pro.k_stride = key_token_stride;
    pro.v_stride = value_token_stride;
    pro.q_stride = rope ? query_token_stride : q_heads * head_dim;
    pro.q_weight = q_weight;
    pro.k_weight = k_weight;
    pro.cos = cos;
    pro.sin = sin;
    pro.q_out = rope ? q_out : nullptr;
    pro.eps = eps;
    return launch_paged_attention(out, query, key_cache, value_cache, block_tables, context_lens, batch,
                                  q_heads, kv_heads, head_dim, num_blocks, block_size, table_width,
                                  partition_tokens, dtype, need, walk, workspace, stream, &pro);
}

extern "C" int mvme_paged_attention_noalloc(void* out, const void* query, const void* key_cache,
                                            const void* value_cache, const int64_t* block_tables,
                                            const int64_t* context_lens, int64_t batch, int64_t q_heads,
                                            int64_t kv_heads, int64_t head_dim, int64_t num_blocks,
                                            int64_t block_size, int64_t table_width, int64_t partition_tokens,
                                            int dtype, void* stream) {
    if (int rc = check_decode_shapes(batch, q_heads, kv_heads, head_dim, num_blocks, block_size,
                                     table_width, dtype))
        return rc;
    if (!out || !query || !key_cache || !value_cache || !block_tables || !context_lens)
        return fail(MVME_EINVAL, "paged attention received a null pointer");
    const bool walk = true;
    const size_t need = mvme_paged_attention_workspace_size(batch, q_heads, kv_heads, head_dim, block_size,
                                                            table_width, partition_tokens);
    if (need > kScratchBytes)
        return fail(MVME_EWORKSPACE, "paged attention (no-alloc) needs " + std::to_string(need) +
                                         " bytes of split-K scratch, above its fixed " +
                                         std::to_string(kScratchBytes) + "; use mvme_paged_attention");
    void* workspace = nullptr;
    if (need > 0)
        if (int rc = device_scratch(&workspace)) return rc;
    return launch_paged_attention(out, query, key_cache, value_cache, block_tables, context_lens, batch,
                                  q_heads, kv_heads, head_dim, num_blocks, block_size, table_width,
                                  partition_tokens, dtype, need, walk, workspace, stream);
}
