// Linear layer for a few rows (the decode batch): out[M, N] = x[M, K] W[N, K]^T
// (+ bias) with nn.Linear's weight layout, for M <= 64, on gfx950 MFMA.
//
// The reference's CudaLinear (mini_engine/kernels/linear.py:14-30) calls
// torch.mm(x, weight.t()); at decode sizes (M = batch, K = N = 2048 for the
// attention output projection) that GEMM reads the 8 MB weight at a small
// fraction of HBM bandwidth, because a library tile sized for large M leaves
// most CUs idle.  Here the weight is the only large operand and is read
// once.  Three kernels:
// * streaming (K = 512, 1024, 1536 or 2048, more than 2048 features: the
//   fused QKV projection, the vocabulary head): persistent work-groups that
//   keep x in registers and stream 16-feature tiles of weight;
// * staged (K a multiple of 512, N of 8, operands within 160 KB of LDS --
//   the decode batch's output projection): one work-group per 8 output
//   features, x and the weight slab copied global->LDS in whole 1 KiB
//   segments;
// * register (any other shape): one work-group per 16 output features, each
//   lane loading its operands straight into registers (by quads where K is a
//   multiple of 128).
// In all, the waves of a work-group split K, each wave computing D[n, m] = W[n, k-slice]
// x[m, k-slice]^T for every 16-row block of x with v_mfma_f32_16x16x32 (fp32
// accumulation), then their partial tiles are summed through LDS and
// rounded once to the output type.  Measured over 28 layers' distinct
// 2048 x 2048 bf16 weights at 32 rows: register kernel 7.8 us per call,
// staged kernel 5.5 us (x re-read from L2 by every work-group dominated the
// register kernel: 5.6 us with the weight loads removed, 4.3 us with the
// x loads removed; with 8 features per work-group, as the staged kernel
// has, it took 7.7 us).
#include <mutex>
#include <type_traits>

#include "mvme_common.h"

namespace mvme {
namespace {

constexpr int kLinWaves = 16;
constexpr int kLinThreads = kLinWaves * kWave;
constexpr int kLinMaxRows = 64;
constexpr int kLinCUs = 256;
constexpr int kStreamMaxK = 2048;  // 16 waves of 128; x's operands for more would not fit the registers

struct LinearArgs {
    void* out;
    const void* x;
    const void* weight;
    const void* bias;  // nullptr: none
    int rows;          // M
    int in_features;   // K, a multiple of 32
    int out_features;  // N, a multiple of 16
    int64_t x_stride;  // elements between rows of x
};

// Sum of NW waves' partials of one (row block, lane) slot of a 16-feature tile,
// every partial read before any is added, and the store of its 4 features.
template <typename T, int NW, typename F>
__device__ inline void sum_and_store(const LinearArgs& a, int n0, int mb, int l, F part) {
    f32x4 p[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) p[w] = part(w);
#pragma unroll
    for (int n = NW; n > 1; n = (n + 1) / 2)
#pragma unroll
        for (int w = 0; w < n / 2; ++w) p[w] += p[w + (n + 1) / 2];
    const int row = 16 * mb + (l & 15);
    if (row >= a.rows) return;
    const int nb = n0 + 4 * (l >> 4);
    float v[4] = {p[0][0], p[0][1], p[0][2], p[0][3]};
    if (a.bias) {
        const uint16_t* bias = static_cast<const uint16_t*>(a.bias) + nb;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] += T::lo((uint32_t)bias[i]);
    }
    const u32x2 packed = {T::pack(v[0], v[1]), T::pack(v[2], v[3])};
    *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(a.out) + (int64_t)row * a.out_features + nb) = packed;
}

// A operand: W rows n0 + (lane % 16), k = k0 + 8 * (lane / 16) .. +8.
// B operand: x rows 16 * mb + (lane % 16), same k.  D: lane holds output
// feature n0 + 4 * (lane / 16) + i (i < 4) for row 16 * mb + lane % 16.
template <typename T, int MB>
__global__ __launch_bounds__(kLinThreads) void linear_rows_kernel(LinearArgs a) {
    __shared__ f32x4 sm_part[kLinWaves][MB][kWave];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const int n0 = blockIdx.x * 16;
    const int li = lane & 15, lg = lane >> 4;
    const int ksteps = a.in_features / 32;
    const uint16_t* wrow = static_cast<const uint16_t*>(a.weight) + (int64_t)(n0 + li) * a.in_features + 8 * lg;
    const uint16_t* xbase = static_cast<const uint16_t*>(a.x) + 8 * lg;
    f32x4 acc[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
    // Rows of x past M read row 0 (in bounds) and are masked to zero.
    bool row_ok[MB];
    const uint16_t* xrow[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        const int r = 16 * mb + li;
        row_ok[mb] = r < a.rows;
        xrow[mb] = xbase + (int64_t)(row_ok[mb] ? r : 0) * a.x_stride;
    }
    // This wave's k-steps: wave, wave + 16, ...  Four in flight at a time (all
    // of them at K = 2048).
    constexpr int kBatch = 4;
    for (int s0 = wave; s0 < ksteps; s0 += kLinWaves * kBatch) {
        u32x4 wv[kBatch], xv[kBatch][MB];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            const int s = min(s0 + j * kLinWaves, ksteps - 1);  // past the end: re-read the last, unused
            wv[j] = *reinterpret_cast<const u32x4*>(wrow + 32 * s);
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) xv[j][mb] = *reinterpret_cast<const u32x4*>(xrow[mb] + 32 * s);
        }
        // No branch between the loads and the products (a branch would make
        // the compiler wait for each step's loads before issuing the next):
        // steps past the end multiply a zero operand.
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            const bool step_ok = s0 + j * kLinWaves < ksteps;
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
                const u32x4 b = (row_ok[mb] && step_ok) ? xv[j][mb] : u32x4{0u, 0u, 0u, 0u};
                acc[mb] = T::mfma16x16x32(wv[j], b, acc[mb]);
            }
        }
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) sm_part[wave][mb][lane] = acc[mb];
    __syncthreads();
    // Thread t sums the waves' partials of one (row block, lane) slot.
    for (int slot = threadIdx.x; slot < MB * kWave; slot += kLinThreads) {
        const int mb = slot / kWave, l = slot % kWave;
        // Every partial is read before any is added (the reads overlap).
        f32x4 part[kLinWaves];
#pragma unroll
        for (int w = 0; w < kLinWaves; ++w) part[w] = sm_part[w][mb][l];
#pragma unroll
        for (int stride = kLinWaves / 2; stride > 0; stride /= 2)
#pragma unroll
            for (int w = 0; w < stride; ++w) part[w] += part[w + stride];
        const f32x4 sum = part[0];
        const int row = 16 * mb + (l & 15);
        if (row >= a.rows) continue;
        const int nb = n0 + 4 * (l >> 4);
        float v[4] = {sum[0], sum[1], sum[2], sum[3]};
        if (a.bias) {
            const uint16_t* bias = static_cast<const uint16_t*>(a.bias) + nb;
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] += T::lo((uint32_t)bias[i]);
        }
        const u32x2 packed = {T::pack(v[0], v[1]), T::pack(v[2], v[3])};
        *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(a.out) + (int64_t)row * a.out_features + nb) = packed;
    }
}

// Register kernel for K a multiple of 128: as above, but with a wave's k-slices
// 128 wide and both operands loaded by quads and transposed (see
// quad_transpose), two slices in flight.  us per call into 2048 features,
// operand-order loads -> quads: K = 4096 10.8 -> 7.8 at 16 rows, 14.7 -> 9.5 at
// 32, 22.7 -> 15.1 at 64; K = 896, 16 rows 5.9 -> 4.1.
template <typename T, int MB>
__global__ __launch_bounds__(kLinThreads) void linear_rows_quads_kernel(LinearArgs a) {
    __shared__ f32x4 sm_part[kLinWaves][MB][kWave];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int n0 = blockIdx.x * 16;
    const int li = lane & 15, lg = lane >> 4;
    const int slices = a.in_features / 128;
    const int quad = li & ~3, chunk = 8 * (4 * lg + (li & 3));
    const uint16_t* wrow = static_cast<const uint16_t*>(a.weight) + (int64_t)(n0 + quad) * a.in_features + chunk;
    const uint16_t* xbase = static_cast<const uint16_t*>(a.x) + chunk;
    f32x4 acc[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
    // F slices from s on, 16 apart, all loaded before the first product.
    auto run = [&](auto count, int s) __attribute__((always_inline)) {
        constexpr int F = decltype(count)::value;
        u32x4 wv[F][4], xv[F][MB][4];
#pragma unroll
        for (int f = 0; f < F; ++f) {
            const int k = 128 * (s + f * kLinWaves);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                wv[f][j] = *reinterpret_cast<const u32x4*>(wrow + (int64_t)j * a.in_features + k);
            // Rows of x past M read row 0 (in bounds); their products are dropped.
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int r = 16 * mb + quad + j;
                    xv[f][mb][j] = *reinterpret_cast<const u32x4*>(xbase + (int64_t)(r < a.rows ? r : 0) * a.x_stride + k);
                }
        }
#pragma unroll
        for (int f = 0; f < F; ++f) {
            quad_transpose(wv[f]);
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
                quad_transpose(xv[f][mb]);
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[mb] = T::mfma16x16x32(wv[f][j], xv[f][mb][j], acc[mb]);
            }
        }
    };
    // (Loading a slice that is not there, to keep one loop, cost depths up to
    // 2048 twice the loads.)
    constexpr int kInFlight = MB <= 2 ? 2 : 1;
    int s = wave;
    for (; s + (kInFlight - 1) * kLinWaves < slices; s += kInFlight * kLinWaves) run(std::integral_constant<int, kInFlight>{}, s);
    if (s < slices) run(std::integral_constant<int, 1>{}, s);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) sm_part[wave][mb][lane] = acc[mb];
    __syncthreads();
    for (int slot = threadIdx.x; slot < MB * kWave; slot += kLinThreads)
        sum_and_store<T, kLinWaves>(a, n0, slot / kWave, slot % kWave,
                                    [&](int w) { return sm_part[w][slot / kWave][slot % kWave]; });
}

// Staged variant for the decode batch (K a multiple of 512, N of 8, x and an
// 8-feature weight slab fitting in LDS): one work-group per 8 output
// features, 256 work-groups at N = 2048, so every CU streams its share of
// the weight.  Both operands reach LDS by direct global->LDS copies of whole
// 1 KiB row segments (coalesced, no VGPR staging): the x rows [16*MB][K]
// with 16-byte chunk c of row r at chunk c ^ (r & 15), the weight rows
// n0..n0+7 [8][K] at c ^ (r & 7), so the operand reads (16 rows x one chunk
// per MFMA) hit distinct banks.  The A operand of the 16x16x32 product
// takes weight row li & 7 (rows 8..15 repeat 0..7; their outputs are
// dropped); each wave then accumulates its k-steps as the register kernel
// does, and the wave partials are summed through LDS (aliasing the x rows).
constexpr int kStagedFeat = 8;
constexpr size_t kStagedMaxLds = 160 * 1024;

__device__ inline void lds_copy16(const void* gptr, uint32_t lds_base) {
    const uint32_t base = __builtin_amdgcn_readfirstlane(lds_base);
    asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(gptr), "s"(base) : "m0");
}

template <typename P>
__device__ inline uint32_t lds_offset(P* p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)p;
}

size_t staged_lds_bytes(int mb, int64_t in_features) {
    const size_t operands = (size_t)(16 * mb + kStagedFeat) * in_features * 2;
    const size_t partials = (size_t)kLinWaves * mb * kWave * sizeof(f32x4);
    return operands > partials ? operands : partials;
}

template <typename T, int MB>
__global__ __launch_bounds__(kLinThreads) void linear_rows_staged_kernel(LinearArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const int n0 = blockIdx.x * kStagedFeat;
    const int li = lane & 15, lg = lane >> 4;
    const int K = a.in_features;
    const int row_chunks = K / 8;          // 16-byte chunks per row
    const int row_instr = row_chunks / 64;  // 1 KiB copies per row
    uint8_t* xs = smem;
    uint8_t* ws = smem + (size_t)16 * MB * K * 2;
    // The weight slab first: its copies come from HBM, x's from L2 (every
    // work-group reads the same x), so the longer latency starts first
    // (5.9 -> 5.5 us per call at 32 x 2048 x 2048).
    for (int i = wave; i < kStagedFeat * row_instr; i += kLinWaves) {
        const int r = i / row_instr, cbase = (i % row_instr) * 64;
        const int c = (cbase + lane) ^ (r & 7);
        const uint16_t* src = static_cast<const uint16_t*>(a.weight) + (int64_t)(n0 + r) * K + 8 * c;
        lds_copy16(src, lds_offset(ws) + (uint32_t)(r * row_chunks + cbase) * 16);
    }
    // Rows of x past M copy row 0 (in bounds); their products are dropped.
    for (int i = wave; i < 16 * MB * row_instr; i += kLinWaves) {
        const int r = i / row_instr, cbase = (i % row_instr) * 64;
        const int c = (cbase + lane) ^ (r & 15);
        const uint16_t* src = static_cast<const uint16_t*>(a.x) + (int64_t)(r < a.rows ? r : 0) * a.x_stride + 8 * c;
        lds_copy16(src, lds_offset(xs) + (uint32_t)(r * row_chunks + cbase) * 16);
    }
    __builtin_amdgcn_s_waitcnt(0);  // this wave's copies landed
    __syncthreads();                // everyone's
    f32x4 acc[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int wr = li & 7;
    for (int st = wave; st < K / 32; st += kLinWaves) {
        const u32x4 w = *reinterpret_cast<const u32x4*>(ws + (size_t)(wr * row_chunks + ((4 * st + lg) ^ wr)) * 16);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            const int r = 16 * mb + li;
            u32x4 x = *reinterpret_cast<const u32x4*>(xs + (size_t)(r * row_chunks + ((4 * st + lg) ^ (r & 15))) * 16);
            if (r >= a.rows) x = u32x4{0u, 0u, 0u, 0u};
            acc[mb] = T::mfma16x16x32(w, x, acc[mb]);
        }
    }
    __syncthreads();  // the operand rows are no longer read
    f32x4* part = reinterpret_cast<f32x4*>(smem);  // [wave][MB][lane]
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) part[(wave * MB + mb) * kWave + lane] = acc[mb];
    __syncthreads();
    // Thread t sums the waves' partials of one (row block, lane) slot whose
    // features are real (lanes 0..31 of the tile hold features 0..7).
    for (int slot = threadIdx.x; slot < MB * kWave; slot += kLinThreads) {
        const int mb = slot / kWave, l = slot % kWave;
        if ((l >> 4) >= kStagedFeat / 4) continue;
        f32x4 p[kLinWaves];
#pragma unroll
        for (int w = 0; w < kLinWaves; ++w) p[w] = part[(w * MB + mb) * kWave + l];
#pragma unroll
        for (int stride = kLinWaves / 2; stride > 0; stride /= 2)
#pragma unroll
            for (int w = 0; w < stride; ++w) p[w] += p[w + stride];
        const int row = 16 * mb + (l & 15);
        if (row >= a.rows) continue;
        const int nb = n0 + 4 * (l >> 4);
        float v[4] = {p[0][0], p[0][1], p[0][2], p[0][3]};
        if (a.bias) {
            const uint16_t* bias = static_cast<const uint16_t*>(a.bias) + nb;
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] += T::lo((uint32_t)bias[i]);
        }
        const u32x2 packed = {T::pack(v[0], v[1]), T::pack(v[2], v[3])};
        *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(a.out) + (int64_t)row * a.out_features + nb) = packed;
    }
}

// Streaming variant for wide layers (the vocabulary head): persistent
// work-groups of NW = K/128 waves, 16 waves per CU, each work-group over a
// contiguous range of 16-feature tiles.  Wave w owns the k-slice [128 w,
// 128 w + 128) and keeps x's operand for it in registers for the whole call
// (16*MB VGPRs), so a tile costs its weight rows and nothing else: two tiles
// of weight loads are in flight per wave (8 KiB, 128 KiB per CU).  The
// waves' partial tiles meet in LDS, double-buffered, with one barrier per
// tile, and MB of the waves (others for the next tile) sum and store it.
// Bound by HBM: 32 rows of 2048 into 151,936 features (622 MB of bf16 weight)
// 314 us with the staged kernel, whose 160 KB of LDS leave one work-group per
// CU with nothing in flight while it multiplies, 105.6 us here (5.9 TB/s).
//
// A product wants 16 features in 16 consecutive lanes; loaded that way,
// every quad of lanes touches four rows and the load unit spends a cycle per
// lane.  Here load j of lane (4*a + p, lg) takes chunk 4*lg + p of feature
// 4*a + j -- a quad reads 64 consecutive bytes -- and a 4x4 transpose inside
// the quads (quad_transpose) turns the four loads into four operands: chunk
// 4*lg + j of feature li.  Same call with operand-order loads 131.9 us.
constexpr int kStreamSteps = 4;  // 32-wide k-steps per wave
// Waves per CU: four per SIMD, three where 64 rows' operands and a work-group
// below 16 waves would otherwise spill.
template <int MB, int NW>
constexpr int stream_waves() { return MB == 4 && NW < kLinWaves ? 12 : 16; }

template <typename T, int MB, int NW>
__global__ __launch_bounds__(NW * kWave, (stream_waves<MB, NW>() / 4)) void linear_rows_stream_kernel(LinearArgs a) {
    __shared__ f32x4 sm_part[2][NW][MB][kWave];
    constexpr int KS = kStreamSteps;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int li = lane & 15, lg = lane >> 4;
    constexpr int K = NW * KS * 32;
    const int tiles = a.out_features / 16;
    const int t_begin = (int)((int64_t)blockIdx.x * tiles / gridDim.x);
    const int t_end = (int)((int64_t)(blockIdx.x + 1) * tiles / gridDim.x);
    if (t_begin >= t_end) return;
    const uint16_t* wbase = static_cast<const uint16_t*>(a.weight) + (int64_t)(li & ~3) * K + wave * (KS * 32) +
                            8 * (4 * lg + (li & 3));
    auto load = [&](int t, u32x4 (&w)[KS]) __attribute__((always_inline)) {
        const uint16_t* p = wbase + (int64_t)min(t, t_end - 1) * (16 * K);
#pragma unroll
        for (int j = 0; j < KS; ++j) w[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p + j * K));
    };
    u32x4 wa[KS], wb[KS];
    load(t_begin, wa);
    // x's operands, loaded and transposed like the weight's (64 rows into 4096
    // features 11.9 -> 9.4 us, 32 rows 7.8 -> 7.0).  Rows past M read row 0 (in
    // bounds); their products are dropped.
    u32x4 xop[MB][KS];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int j = 0; j < KS; ++j) {
            const int r = 16 * mb + (li & ~3) + j;
            xop[mb][j] = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(a.x) +
                                                         (int64_t)(r < a.rows ? r : 0) * a.x_stride +
                                                         wave * (KS * 32) + 8 * (4 * lg + (li & 3)));
        }
    load(t_begin + 1, wb);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) quad_transpose(xop[mb]);
    auto tile = [&](int t, u32x4 (&w)[KS], int buf) __attribute__((always_inline)) {
        f32x4 acc[MB];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
        quad_transpose(w);
#pragma unroll
        for (int j = 0; j < KS; ++j)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) acc[mb] = T::mfma16x16x32(w[j], xop[mb][j], acc[mb]);
        load(t + 2, w);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) sm_part[buf][wave][mb][lane] = acc[mb];
        // One barrier per tile: it publishes this tile's partials, and the
        // sums of the tile before the last (this buffer's previous use) were
        // read before their waves came to the previous barrier.
        __syncthreads();
        // Wave w sums row block mb when w = (t - t_begin) * MB + mb (mod NW).
        const int first = (t - t_begin) * MB % NW;
        const int mb = wave >= first ? wave - first : wave - first + NW;
        if (mb >= MB) return;
        sum_and_store<T, NW>(a, 16 * t, mb, lane, [&](int w) { return sm_part[buf][w][mb][lane]; });
    };
    // Pairs without a branch between the two tiles: with one, the compiler's
    // wait for the first tile's weights also covers the second's.
    int t = t_begin;
    for (; t + 1 < t_end; t += 2) {
        tile(t, wa, 0);
        tile(t + 1, wb, 1);
    }
    if (t < t_end) tile(t, wa, 0);
}

template <typename T, int MB, int NW>
void launch_stream(const LinearArgs& a, hipStream_t s) {
    const int groups = min(a.out_features / 16, kLinCUs * (stream_waves<MB, NW>() / NW));
    hipLaunchKernelGGL((linear_rows_stream_kernel<T, MB, NW>), dim3(groups), dim3(NW * kWave), 0, s, a);
}

template <typename T, int MB>
void launch_stream_nw(const LinearArgs& a, hipStream_t s) {
    switch (a.in_features / (32 * kStreamSteps)) {
        case 4: launch_stream<T, MB, 4>(a, s); break;
        case 8: launch_stream<T, MB, 8>(a, s); break;
        case 12: launch_stream<T, MB, 12>(a, s); break;
        default: launch_stream<T, MB, 16>(a, s); break;
    }
}

template <typename T>
void launch_linear_stream(const LinearArgs& a, int mb, hipStream_t s) {
    if (mb == 1) launch_stream_nw<T, 1>(a, s);
    else if (mb == 2) launch_stream_nw<T, 2>(a, s);
    else if (mb == 3) launch_stream_nw<T, 3>(a, s);
    else launch_stream_nw<T, 4>(a, s);
}

template <typename T, int MB>
int launch_staged(const LinearArgs& a, hipStream_t s) {
    const size_t lds = staged_lds_bytes(MB, a.in_features);
    static std::once_flag once;
    static hipError_t attr = hipSuccess;
    std::call_once(once, [] {
        attr = hipFuncSetAttribute(reinterpret_cast<const void*>(linear_rows_staged_kernel<T, MB>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)kStagedMaxLds);
    });
    if (attr != hipSuccess) return fail(MVME_ELAUNCH, std::string("linear rows: LDS size attribute: ") +
                                                      hipGetErrorString(attr));
    hipLaunchKernelGGL((linear_rows_staged_kernel<T, MB>), dim3((unsigned)(a.out_features / kStagedFeat)),
                       dim3(kLinThreads), lds, s, a);
    return MVME_OK;
}

template <typename T>
int launch_linear_staged(const LinearArgs& a, int mb, hipStream_t s) {
    if (mb == 1) return launch_staged<T, 1>(a, s);
    if (mb == 2) return launch_staged<T, 2>(a, s);
    if (mb == 3) return launch_staged<T, 3>(a, s);
    return launch_staged<T, 4>(a, s);
}

template <typename T>
void launch_linear_rows(const LinearArgs& a, hipStream_t s) {
    const dim3 grid((unsigned)(a.out_features / 16)), block(kLinThreads);
    const int mb = (a.rows + 15) / 16;
    // One to three rows into wide layers keep operand-order loads, whose x is then one
    // to three lines and whose 16 waves all work at any depth.  us per call, operand
    // order / quads: 1 row, K = 4096, N = 8192 14.6 / 16.0, K = 1920, N = 16384 14.2 /
    // 15.9; 3 rows 15.3 / 16.1, 14.8 / 16.0; 6 rows 16.7 / 16.1; 1 row, K = 4096, N =
    // 6144 14.4 / 14.5, K = 1408, N = 16384 14.1 / 14.0, K = 5120, N = 8192 19.0 / 17.5.
    const bool few_rows = a.rows <= 3 && a.out_features >= 8192 && a.in_features > 1536 && a.in_features <= 4096;
    if (a.in_features % 128 == 0 && !few_rows) {
        if (mb == 1) hipLaunchKernelGGL((linear_rows_quads_kernel<T, 1>), grid, block, 0, s, a);
        else if (mb == 2) hipLaunchKernelGGL((linear_rows_quads_kernel<T, 2>), grid, block, 0, s, a);
        else if (mb == 3) hipLaunchKernelGGL((linear_rows_quads_kernel<T, 3>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((linear_rows_quads_kernel<T, 4>), grid, block, 0, s, a);
        return;
    }
    if (mb == 1) hipLaunchKernelGGL((linear_rows_kernel<T, 1>), grid, block, 0, s, a);
    else if (mb == 2) hipLaunchKernelGGL((linear_rows_kernel<T, 2>), grid, block, 0, s, a);
    else if (mb == 3) hipLaunchKernelGGL((linear_rows_kernel<T, 3>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((linear_rows_kernel<T, 4>), grid, block, 0, s, a);
}

}  // namespace
}  // namespace mvme

using namespace mvme;

extern "C" int mvme_linear_rows(void* out, const void* x, const void* weight, const void* bias, int64_t rows,
                                int64_t in_features, int64_t out_features, int64_t x_row_stride, int dtype,
                                void* stream) {
    if (dtype != MVME_FP16 && dtype != MVME_BF16) return fail(MVME_EINVAL, "linear rows supports FP16/BF16");
    if (rows < 0 || rows > kLinMaxRows) return fail(MVME_EINVAL, "linear rows supports at most 64 rows");
    if (in_features <= 0 || in_features % 32 != 0 || in_features > 2147483647)
        return fail(MVME_EINVAL, "linear rows needs in_features a positive multiple of 32");
    if (out_features <= 0 || out_features % 16 != 0 || out_features / 16 > 2147483647)
        return fail(MVME_EINVAL, "linear rows needs out_features a positive multiple of 16");
    if (x_row_stride < in_features || x_row_stride % 8 != 0)
        return fail(MVME_EINVAL, "linear rows needs a row stride >= in_features and a multiple of 8");
    if (rows == 0) return MVME_OK;
    if (!out || !x || !weight) return fail(MVME_EINVAL, "linear rows received a null pointer");
    const auto misaligned = [](const void* p, uintptr_t m) { return (reinterpret_cast<uintptr_t>(p) & m) != 0; };
    if (misaligned(x, 15) || misaligned(weight, 15) || misaligned(out, 7) || (bias && misaligned(bias, 1)))
        return fail(MVME_EINVAL, "linear rows needs 16-byte aligned x and weight and 8-byte aligned out");
    LinearArgs a{};
    a.out = out;
    a.x = x;
    a.weight = weight;
    a.bias = bias;
    a.rows = (int)rows;
    a.in_features = (int)in_features;
    a.out_features = (int)out_features;
    a.x_stride = x_row_stride;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int mb = (int)((rows + 15) / 16);
    // More features than one round of staged work-groups (8 each, one per CU)
    // stream; at most that many fit the chip at once and start faster staged
    // (no prologue that loads x into registers).  us per call, staged against
    // streaming, K = 2048: N = 2048 4.3 / 5.3 at 16 rows, 5.7 / 6.9 at 32;
    // N = 4096 8.3 / 6.1, 10.6 / 7.0, 13.2 / 9.4 at 64; N = 8192 14.3 / 11.0;
    // K = 1024, N = 4096 4.4 / 4.2.
    if (in_features % 512 == 0 && in_features <= kStreamMaxK && out_features > kLinCUs * kStagedFeat) {
        if (dtype == MVME_FP16) launch_linear_stream<Half>(a, mb, s);
        else launch_linear_stream<BFloat16>(a, mb, s);
        return check_launch("linear rows");
    }
    if (in_features % 512 == 0 && out_features % kStagedFeat == 0 &&
        staged_lds_bytes(mb, in_features) <= kStagedMaxLds) {
        const int rc = dtype == MVME_FP16 ? launch_linear_staged<Half>(a, mb, s) : launch_linear_staged<BFloat16>(a, mb, s);
        if (rc != MVME_OK) return rc;
        return check_launch("linear rows");
    }
    if (dtype == MVME_FP16) launch_linear_rows<Half>(a, s);
    else launch_linear_rows<BFloat16>(a, s);
    return check_launch("linear rows");
}
