// Projections over f16 weights: Y = X W^T (+ bias), optionally RMS-normalized input, accumulate, f16 output.
//
// Reference behaviour (dooms.cpp 0.6.1, src/backend/metal/llama_kernels.h):
//   * matvec1 (96-126) / matvecm (809-842), one to eight tokens: f32 input rows, y = (W . (x * gamma)) * scale + bias,
//     scale = 1 / sqrt(sum x^2 / K + eps) reduced over the row (stage_input, 62-80);
//   * matmul / matmul_big (222-255, 418-450), prompt chunks: the input tile staged as half(x * gamma * scale) with the
//     row scale from rms_scale (312-328), half x half products accumulated in f32, then + bias, or added into y.
//   * the Whisper cross-attention cache: matmul_big into an f32 scratch, then to_half (metal_whisper_decoder.mm:295-316);
//     here the GEMM rounds to half in its epilogue and writes the cache row directly.
//
// MI355X design:
//   * M <= 8 (decode): gemv_kernel, HBM-bound on the weights (2 N K bytes, each read once). One workgroup per CU
//     (1 to 8 waves, as the rows divide) stages the (normalized) input rows in LDS once; each wave owns 2 or 4 weight rows and
//     streams them in 16-byte non-temporal loads (the weights are read once per step; the cache lines are not kept:
//     q|k|v 12.9 -> 11.7 us, attn_output 10.1 -> 9.3 us, a 14336-column down projection 26.0 -> 23.2 us), 4 sweeps
//     (8 with eight input rows) of 2 or 4 loads in flight per lane. The input rows' loads go out first, in one
//     batch, then the first sweeps of weight loads, so that the staging waits only for the input; the dot products
//     stay f32 and are reduced across the wave at the end.
//   * M > 8 (prompt, batched decode): stage_kernel writes each input row once as half(x * gamma * scale) into the
//     workspace (the reference stages the same values per tile). Products with enough tiles for every CU run on
//     gemm_big_tile, 256-row tiles of 8 waves; the others on gemm_split_tile, smaller tiles and K cut into parts, so
//     that a product of few rows streams its weights through the whole chip. linear_plan picks by a fitted cost.
//   * Several matrices with the same input and shape (the cross cache's K and V of every layer) run in one launch.
//   * mx_linear runs these kernels only: no vendor GEMM library is loaded or linked.

#include <algorithm>
#include <type_traits>

#include "linear_plan.hpp"
#include "mx_common.hpp"
#include "mx_kernels.hpp"

namespace mx {

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;

// ---- M > 8: the input rows staged once as half, as the reference's matmul staging does per tile
// (half(x * gamma * rms_scale), llama_kernels.h:186-199, with rms_scale from llama_kernels.h:312-328): one workgroup
// per row; the GEMM then multiplies half operands only ----
template <bool NORM>
__global__ __launch_bounds__(kThreads) void stage_kernel(LinearParams p) {
    __shared__ float red[kWaves];
    if (p.plan.splits > 1)  // the split GEMM's counters (one per thread of the whole grid; the grid has rows > 8)
        for (int i = blockIdx.x * kThreads + threadIdx.x; i < p.plan.tiles; i += gridDim.x * kThreads)
            p.counters[i * kCounterStride] = 0u;
    const float * row = p.x + (int64_t)blockIdx.x * p.x_stride;
    const int kp = (p.K + 63) / 64 * 64;  // staged rows are zero-padded to a multiple of 64 columns
    half_t * dst = p.xh + (int64_t)blockIdx.x * kp;
    const int K4 = p.K / 4;
    constexpr int SJ = 8;  // 16-byte pieces per thread held in registers
    if (K4 <= SJ * kThreads) {
        // the row (and gamma) loaded once, all pieces in flight together; the sum of squares and the conversion then
        // work from registers
        float4_t v[SJ], g[SJ];
#pragma unroll
        for (int j = 0; j < SJ; j++) {
            const int kk = min(j * kThreads + (int)threadIdx.x, K4 - 1);
            v[j] = *reinterpret_cast<const float4_t *>(row + 4 * kk);
            if constexpr (NORM) g[j] = *reinterpret_cast<const float4_t *>(p.gamma + 4 * kk);
        }
        float s = 1.f;
        if constexpr (NORM) {
            float ss = 0.f;
#pragma unroll
            for (int j = 0; j < SJ; j++)
                if (j * kThreads + (int)threadIdx.x < K4)
                    ss += v[j][0] * v[j][0] + v[j][1] * v[j][1] + v[j][2] * v[j][2] + v[j][3] * v[j][3];
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) ss += shfl_xor(ss, o);
            if (threadIdx.x % kWave == 0) red[threadIdx.x / kWave] = ss;
            __syncthreads();
            float t = 0.f;
#pragma unroll
            for (int w = 0; w < kWaves; w++) t += red[w];
            s = 1.f / __builtin_sqrtf(t / (float)p.K + p.eps);
        }
#pragma unroll
        for (int j = 0; j < SJ; j++) {
            const int kk = j * kThreads + (int)threadIdx.x;
            if (kk >= K4) continue;
            half4_t h;
#pragma unroll
            for (int e = 0; e < 4; e++) h[e] = (half_t)(NORM ? v[j][e] * (g[j][e] * s) : v[j][e]);
            *reinterpret_cast<half4_t *>(dst + 4 * kk) = h;
        }
        for (int k = p.K + threadIdx.x * 8; k < kp; k += kThreads * 8) *reinterpret_cast<u32x4 *>(dst + k) = u32x4{0u, 0u, 0u, 0u};
        return;
    }
    float s = 1.f;
    if constexpr (NORM) {
        float ss = 0.f;
        for (int k = threadIdx.x * 4; k < p.K; k += kThreads * 4) {
            const float4_t v = *reinterpret_cast<const float4_t *>(row + k);
            ss += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) ss += shfl_xor(ss, o);
        if (threadIdx.x % kWave == 0) red[threadIdx.x / kWave] = ss;
        __syncthreads();
        float t = 0.f;
#pragma unroll
        for (int w = 0; w < kWaves; w++) t += red[w];
        s = 1.f / __builtin_sqrtf(t / (float)p.K + p.eps);
    }
    for (int k = threadIdx.x * 8; k < p.K; k += kThreads * 8) {
        float x[8];
        load8f(row + k, x);
        if constexpr (NORM) {
            float g[8];
            load8f(p.gamma + k, g);
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] *= g[e] * s;  // x * (gamma * scale), as the reference's staging
        }
        *reinterpret_cast<u32x4 *>(dst + k) = to_half8(x);
    }
    for (int k = p.K + threadIdx.x * 8; k < kp; k += kThreads * 8) *reinterpret_cast<u32x4 *>(dst + k) = u32x4{0u, 0u, 0u, 0u};
}

// Epilogue of the tiled GEMMs: the lane's 16 outputs of column n of an MFMA tile (rows mbase + 8 (v / 4) + v % 4),
// y (+)= acc (+ bias). The bias and the previous outputs are all loaded before the first
// store: a store to y may alias them as far as the compiler can tell, so with loads and stores interleaved each
// element waited for one or two memory round trips in turn. Rows past M read row M - 1 (a valid address) and store
// nothing.
template <bool OUT16>
__device__ __forceinline__ void store_col16(const LinearParams & p, int mi, int n, int mbase, const float16_t & acc) {
    const float * b = (p.flags & kLinearBias) ? p.bias[mi] : nullptr;
    const float bv = b ? b[n] : 0.f;
    const bool accum = p.flags & kLinearAccumulate;
    float prev[16];
    if (accum) {
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int m = min(mbase + 8 * (v / 4) + v % 4, p.M - 1);
            const int64_t o = (int64_t)m * p.y_stride + n;
            if constexpr (OUT16) prev[v] = (float)static_cast<const half_t *>(p.y[mi])[o];
            else prev[v] = static_cast<const float *>(p.y[mi])[o];
        }
    }
    // every sum before the first store, so that no loaded value is used behind a store (the compiler's waits at the
    // stores' branches would otherwise drain the stores before it)
    float x[16];
#pragma unroll
    for (int v = 0; v < 16; v++) {
        x[v] = acc[v];
        if (b) x[v] += bv;
        if (accum) x[v] += prev[v];
    }
#pragma unroll
    for (int v = 0; v < 16; v++) {
        const int m = mbase + 8 * (v / 4) + v % 4;
        if (m >= p.M) continue;
        const int64_t o = (int64_t)m * p.y_stride + n;
        if constexpr (OUT16) static_cast<half_t *>(p.y[mi])[o] = (half_t)x[v];
        else static_cast<float *>(p.y[mi])[o] = x[v];
    }
}

// ---- M <= 8: f32 input rows in LDS, 2 or 4 weight rows per wave ----
constexpr int kGemvRows = 4;       // weight rows per wave (the most)
constexpr int kGemvMaxWaves = 8;   // waves per workgroup (the launch sizes workgroups so that each CU gets one)
// 64-lane sweeps of 16-byte weight loads in flight per wave: 4, and 8 with eight input rows (more arithmetic per
// weight byte; Llama-3-8B attention output at 8 rows 19.7 -> 17.2 us, while at 1, 2 and 4 rows 8 sweeps were 3-25 %
// slower than 4)
template <int MT>
constexpr int gemv_depth() { return MT == 8 ? 8 : 4; }

// STAGE: the input rows (times gamma) fit the LDS budget and are staged once; otherwise every wave reads them from
// L2 as it goes (the reference's kStageInput = false variant, metal_llama_decoder.mm:45-47).
// The wave's first gemv_depth sweeps of weight loads are issued before the input is staged, so the staging and its
// barriers overlap the first HBM round trip.
template <int MT, bool STAGE, bool OUT16, bool NORM, int RW>
__global__ __launch_bounds__(kGemvMaxWaves * kWave) void gemv_kernel(LinearParams p) {
    extern __shared__ float xs[];  // [MT][K]: x (* gamma) of each input row, when staged
    __shared__ float red[MT][kGemvMaxWaves];
    __shared__ float s_scale[MT];
    constexpr int kGemvDepth = gemv_depth<MT>();
    const int K = p.K, M = p.M;
    constexpr bool norm = NORM;  // p.flags & kLinearNorm
    const int nw = blockDim.x / kWave;
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;

    // work item: (matrix, group of RW rows) per wave
    const int groups = (p.N + RW - 1) / RW;
    const int item = __builtin_amdgcn_readfirstlane(blockIdx.x * nw + wave);  // wave-uniform: scalar loads of p.w[mi]
    const bool active = item < groups * p.count;
    const int mi = active ? item / groups : 0;
    const int r0 = active ? (item % groups) * RW : 0;
    const half_t * w = p.w[mi];
    const half_t * wr[RW];
#pragma unroll
    for (int i = 0; i < RW; i++) wr[i] = w + (int64_t)min(r0 + i, p.N - 1) * K;
    const int C8 = K / 8;  // 16-byte chunks per row
    half8_t wv[kGemvDepth][RW];
    auto load_sweep = [&](int j, int c) __attribute__((always_inline)) {
        const int cc = min(c, C8 - 1);  // past the row: a valid chunk, not used
#pragma unroll
        for (int i = 0; i < RW; i++)  // non-temporal: each weight is read once per step
            wv[j][i] = as_half8(__builtin_nontemporal_load((const __attribute__((address_space(1))) u32x4 *)(wr[i] + 8 * cc)));
    };

    // The input rows (and gamma) in batches: batch b covers the 16-byte chunks kk = (b XJ + j) blockDim + tid, j < XJ,
    // of every input row. All of a batch's loads go out before any wait (clamped, unconditional), and batch 0 goes out
    // ahead of the weight loads: loads complete in issue order, so its wait leaves the weights in flight.
    constexpr int XJ = MT >= 4 ? 1 : 4 / MT;
    const int K4 = K / 4;
    const int nxb = (STAGE || NORM) ? (K4 + XJ * (int)blockDim.x - 1) / (XJ * (int)blockDim.x) : 0;
    float4_t xv[MT][XJ], gv[XJ];
    float ss[MT];
#pragma unroll
    for (int m = 0; m < MT; m++) ss[m] = 0.f;
    auto xload = [&](int b) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < XJ; j++) {
            const int kk = min((b * XJ + j) * (int)blockDim.x + (int)threadIdx.x, K4 - 1);
            if constexpr (NORM) gv[j] = *reinterpret_cast<const float4_t *>(p.gamma + 4 * kk);
#pragma unroll
            for (int m = 0; m < MT; m++)
                xv[m][j] = *reinterpret_cast<const float4_t *>(p.x + (int64_t)min(m, M - 1) * p.x_stride + 4 * kk);
        }
    };
    // sums of squares (stage_input, llama_kernels.h:62-80) and the staged x (* gamma)
    auto xstage = [&](int b) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < XJ; j++) {
            const int kk = (b * XJ + j) * (int)blockDim.x + (int)threadIdx.x;
            if (kk >= K4) continue;
#pragma unroll
            for (int m = 0; m < MT; m++) {
                const float4_t v = xv[m][j];
                if constexpr (NORM) ss[m] += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
                if constexpr (STAGE)
                    if (m < M) *reinterpret_cast<float4_t *>(xs + m * K + 4 * kk) = NORM ? v * gv[j] : v;
            }
        }
    };
    if constexpr (STAGE || NORM) xload(0);
    __builtin_amdgcn_sched_barrier(0);  // keep the issue order: the input first, then the weights
    // unconditional (an idle wave reads valid rows of matrix 0 and returns below): a branch here would make every
    // later wait assume that the input loads are the newest ones
#pragma unroll
    for (int j = 0; j < kGemvDepth; j++) load_sweep(j, lane + kWave * j);
    // what the epilogue adds to lane i MT + m's output (row r0 + i, input row m): the bias and the previous output,
    // loaded here behind the weights (by every lane, at clamped valid addresses) rather than after the reduction,
    // where each was one more memory round trip at the end of the kernel
    float y_prev = 0.f, y_bias = 0.f;
    {
        const int i = min(lane / MT, RW - 1), m = min(lane % MT, M - 1), n = min(r0 + i, p.N - 1);
        if (p.flags & kLinearAccumulate) {
            const int64_t o = (int64_t)m * p.y_stride + n;
            if constexpr (OUT16) y_prev = (float)static_cast<const half_t *>(p.y[mi])[o];
            else y_prev = static_cast<const float *>(p.y[mi])[o];
        }
        if (p.flags & kLinearBias) {
            const float * b = p.bias[mi];
            if (b) y_bias = b[n];
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (STAGE || NORM) xstage(0);
    for (int b = 1; b < nxb; b++) {  // inputs longer than one batch (the waits of these drain the weight loads too)
        xload(b);
        xstage(b);
        // nothing in flight after the loop (else the compiler, for a register whose load may still be pending past
        // the loop, drains every weight load ahead of the sweeps, also where the loop never runs: q|k|v 11.85 ->
        // 11.11 us, Whisper attention output 3.64 -> 3.38)
        __builtin_amdgcn_s_waitcnt(0);
    }
    if (norm) {
#pragma unroll
        for (int m = 0; m < MT; m++) {
            float t = ss[m];
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) t += shfl_xor(t, o);
            if (lane == 0) red[m][wave] = t;
        }
    }
    __syncthreads();
    if (norm && threadIdx.x < MT) {
        float t = 0.f;
        for (int w2 = 0; w2 < nw; w2++) t += red[threadIdx.x][w2];
        s_scale[threadIdx.x] = 1.f / __builtin_sqrtf(t / (float)K + p.eps);
    }
    __syncthreads();
    if (!active) return;  // after the last barrier

    float acc[RW][MT];
#pragma unroll
    for (int i = 0; i < RW; i++)
#pragma unroll
        for (int m = 0; m < MT; m++) acc[i][m] = 0.f;
    auto sweep = [&](int j, int c) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < MT; m++) {
            float4_t x0, x1;
            if constexpr (STAGE) {
                x0 = *reinterpret_cast<const float4_t *>(xs + m * K + 8 * c);
                x1 = *reinterpret_cast<const float4_t *>(xs + m * K + 8 * c + 4);
            } else {
                const float * xr = p.x + (int64_t)min(m, M - 1) * p.x_stride + 8 * c;
                x0 = *reinterpret_cast<const float4_t *>(xr);
                x1 = *reinterpret_cast<const float4_t *>(xr + 4);
                if (norm) {
                    x0 = x0 * *reinterpret_cast<const float4_t *>(p.gamma + 8 * c);
                    x1 = x1 * *reinterpret_cast<const float4_t *>(p.gamma + 8 * c + 4);
                }
            }
#pragma unroll
            for (int i = 0; i < RW; i++) {
                float a = acc[i][m];
#pragma unroll
                for (int e = 0; e < 4; e++) a = __builtin_fmaf((float)wv[j][i][e], x0[e], a);
#pragma unroll
                for (int e = 0; e < 4; e++) a = __builtin_fmaf((float)wv[j][i][4 + e], x1[e], a);
                acc[i][m] = a;
            }
        }
    };
    // sweep j of pass q covers chunk 256 q + 64 j + lane; its registers are reloaded for the next pass right after use.
    // The loads are unconditional inside the loop and the last pass is peeled off (no loads), so the compiler's waits
    // track each sweep's own loads instead of draining every load at the top of a pass.
    constexpr int kPass = kWave * kGemvDepth;
    const int npass = (C8 + kPass - 1) / kPass;
    for (int q = 0; q + 1 < npass; q++) {
#pragma unroll
        for (int j = 0; j < kGemvDepth; j++) {
            const int c = q * kPass + kWave * j + lane;  // < C8: not the last pass
            sweep(j, c);
            load_sweep(j, c + kPass);
        }
    }
#pragma unroll
    for (int j = 0; j < kGemvDepth; j++) {
        const int c = (npass - 1) * kPass + kWave * j + lane;
        if (c < C8) sweep(j, c);
    }
    // reduce over the wave; lane i * MT + m stores (row r0 + i, input row m)
    float mine = 0.f;
#pragma unroll
    for (int i = 0; i < RW; i++)
#pragma unroll
        for (int m = 0; m < MT; m++) {
            const float s = wave_sum(acc[i][m]);
            if (lane == i * MT + m) mine = s;
        }
    if (lane < RW * MT) {
        const int i = lane / MT, m = lane % MT, n = r0 + i;
        if (m < M && n < p.N) {  // the bias and the previous output loaded above
            float v = norm ? mine * s_scale[m] : mine;
            if (p.flags & kLinearBias) v += y_bias;
            if (p.flags & kLinearAccumulate) v += y_prev;
            const int64_t o = (int64_t)m * p.y_stride + n;
            if constexpr (OUT16) static_cast<half_t *>(p.y[mi])[o] = (half_t)v;
            else static_cast<float *>(p.y[mi])[o] = v;
        }
    }
}

// ---- M > 8, large products: 256 x 256 tiles of 8 waves (each 128 x 64, 4 x 2 MFMA tiles), K in steps of 64 ----
// A 128 x 128 tile streams 64 bytes per clock and CU from L2 at the MFMA rate, the whole of an XCD's L2 bandwidth;
// 256 x 256 halves the bytes per product (and 128 x 64 per wave cuts the LDS reads per product by a quarter). The
// tiles go from HBM/L2 straight into LDS (global_load_lds_dwordx4: lane l's 16 bytes land at byte 16 l of the
// instruction's 1 KB destination), two buffers (the loads of step s + 1 in flight while step s multiplies), no
// registers in between. A load covers 8 rows x 128 bytes, whole cache lines: in pieces of 64 bytes every line came to
// the CU twice. 16-byte chunk c of row r sits at 16 (c ^ (r / 2 % 8)) within its row's 128 bytes, so the 16-byte operand
// reads of 16 consecutive rows at one chunk land on 16 distinct 4-bank groups. 128 KB of LDS: one workgroup per CU,
// two waves per SIMD, which take turns (below). The load path bounds it: without the loads 2048 x 6144 x 4096 takes
// 102 us instead of 130, without most of the products 105, without half of the operand reads no less. Against one barrier per
// step, both waves of a SIMD in step and 64-byte pieces (us, staging included, one box): 2048 x 6144 x 4096 140 -> 130,
// 4096 x 4096 x 4096 175 -> 158, 8 products of 1500 x 1280 x 1280 62.8 -> 55.7, 1024 x 14336 x 4096 150 -> 136, 3000 x 4096 x
// 14336 445 -> 392. The raised wave priority around the products, the loads all in the first phase, spread over all
// four or ahead of the operand reads, and phases of two slices measured 1 to 10 % slower.
// BN = 192 (256 x 192, 8 waves of 64 x 96) serves products whose 256 x 256 tiles would leave CUs idle.
constexpr int kBM = kGemmBigRows;
constexpr int kBigWaves = 8, kBigThreads = kBigWaves * kWave;
// WC: columns per wave (64, or 96 for 256 x 192 tiles: 8 waves of 64 x 96).
// HALF: K is an odd multiple of 32. The staged rows are zero-padded to the last step's 64 columns, the chunks past the
// weights' row read the four before them, and the last step's second half takes no part in the products (zeros of the
// staged rows would make NaN of an infinity). Walked in 32-column steps through three buffers, 2048 x 6144 x 4128 took
// 131 us, on 128-row tiles 138, so 117 (3000 x 4096 x 14304 445, 501 and 426).
template <bool OUT16, int BN, int WC, bool HALF>
__device__ __forceinline__ void gemm_big_tile(const LinearParams & p) {
    constexpr int kBN = BN, kBK = 64;
    constexpr int kBlocks = (kBM + BN) / 8;                  // 1 KB blocks (8 rows x 128 bytes) of a step's tiles
    constexpr int Loads = kBlocks / kBigWaves;               // direct loads per wave and step
    constexpr int WN = BN / WC, WM = kBigWaves / WN;         // waves along N and along M
    constexpr int kBigMI = kBM / WM / 32, kBigNJ = WC / 32;  // 32 x 32 MFMA tiles per wave
    static_assert(kBlocks % kBigWaves == 0 && kBigMI >= 1 && WN * WM == kBigWaves, "whole loads and tiles per wave");
    __shared__ __attribute__((aligned(1024))) half_t sm[2][(kBM + BN) * kBK];  // A's rows, then B's
    const int n_tiles = (p.N + kBN - 1) / kBN, m_tiles = (p.M + kBM - 1) / kBM;
    // consecutive work items share a weight tile (different token tiles); contiguous ranges per XCD
    const uint32_t t = xcd_remap(blockIdx.x, (uint32_t)(p.count * n_tiles * m_tiles));
    const int mt = t % m_tiles, nt = (t / m_tiles) % n_tiles, mi = t / (m_tiles * n_tiles);
    const int m0 = mt * kBM, n0 = nt * kBN;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    const int l32 = lane % 32, hi = lane / 32;

    // Each lane's source bytes relative to the step's first column are fixed: rows past M (N) repeat the last row. The
    // staged rows are K rounded up to 64 halves apart. Lane l of block j fills position l % 8 of the tile's row
    // 8 j + l / 8 with 16-byte chunk (l % 8) ^ (row / 2 % 8).
    const int kp = HALF ? p.K + 32 : p.K, nk = kp / kBK;
    const char * a_base = reinterpret_cast<const char *>(p.xh + (int64_t)m0 * kp);
    const char * b_base = reinterpret_cast<const char *>(p.w[mi] + (int64_t)n0 * p.K);
    uint32_t off[Loads];
#pragma unroll
    for (int i = 0; i < Loads; i++) {
        const int j = i * kBigWaves + wave, row = gemm_block_row<kBK>(j, lane), chunk = gemm_block_chunk<kBK>(j, lane);
        off[i] = row < kBM ? gemm_load_offset<uint32_t>(m0, row, p.M, kp, chunk)
                           : gemm_load_offset<uint32_t>(n0, row - kBM, p.N, p.K, chunk);
    }
    // HALF: what this lane's weight loads of the last step go back (kBigWaves is even: every block of a wave has its swizzle)
    const uint32_t back = HALF ? gemm_half_back(gemm_block_chunk<kBK>(wave, lane)) : 0;
    // loads I0 .. I1 - 1 of a step
    auto issue = [&](int step, auto I0C, auto I1C) __attribute__((always_inline)) {
        const int64_t k0 = (int64_t)step * kBK * 2;  // bytes
        static_for<decltype(I0C)::value, decltype(I1C)::value>([&](auto I) __attribute__((always_inline)) {
            constexpr int i = decltype(I)::value;
            constexpr bool a = i * kBigWaves < kBM / 8;
            const int j = i * kBigWaves + wave;
            const uint32_t o = HALF && !a && step == nk - 1 ? off[i] - back : off[i];
            __builtin_amdgcn_global_load_lds((a ? a_base : b_base) + k0 + o,
                                             (__attribute__((address_space(3))) void *)&sm[step & 1][512 * j], 16, 0, 0);
        });
    };
    static_assert(kBM / 8 % kBigWaves == 0, "a load is of A or of B for every wave");

    float16_t acc[kBigMI][kBigNJ];
#pragma unroll
    for (int i = 0; i < kBigMI; i++)
#pragma unroll
        for (int j = 0; j < kBigNJ; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;

    // this wave's block: rows (256 / WM) wm + 32 i + l32 of A, columns WC wn + 32 j + l32 (rows of B); fragment (row,
    // chunk 2 ks + hi) at byte 128 row + 16 ((2 ks + hi) ^ (row / 2 % 8))
    const int wm = wave / WN, wn = wave % WN;
    uint32_t rd[4];
#pragma unroll
    for (int ks = 0; ks < 4; ks++) rd[ks] = 128 * l32 + 16 * ((2 * ks + hi) ^ ((l32 >> 1) & 7));
    const uint32_t sm0 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) half_t *)sm[0];
    auto barrier = []() __attribute__((always_inline)) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
    };
    using I0 = std::integral_constant<int, 0>;
    using IH = std::integral_constant<int, Loads / 2>;
    using IE = std::integral_constant<int, Loads>;
    issue(0, I0{}, IE{});
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    barrier();
    // Waves 4 .. 7 run half a phase behind waves 0 .. 3: of the two waves of a SIMD one multiplies while the other reads its
    // operands and issues loads. A phase is a 16-column slice of a step: the slice's operand reads (and in phases 0 and
    // 1 the next step's loads), a barrier, its products, a barrier.
    const bool behind = wave >= kBigWaves / 2;
    if (behind) barrier();
    for (int s = 0; s < nk; s++) {
        const uint32_t xa = sm0 + (uint32_t)(s & 1) * ((kBM + BN) * kBK * 2) + 128 * (kBM / WM) * wm;
        const uint32_t wa = sm0 + (uint32_t)(s & 1) * ((kBM + BN) * kBK * 2) + 128 * (kBM + WC * wn);
        static_for<0, 4>([&](auto KS) __attribute__((always_inline)) {
            constexpr int ks = decltype(KS)::value;
            // the operand reads as inline asm (the compiler cannot tell them from the direct loads in flight, and would
            // wait for those)
            u32x4 fa[kBigMI], fb[kBigNJ];
            static_for<0, kBigNJ>([&](auto J) __attribute__((always_inline)) {
                u32x4 r;
                asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(wa + rd[ks]), "i"(4096 * decltype(J)::value));
                fb[decltype(J)::value] = r;
            });
            static_for<0, kBigMI>([&](auto I) __attribute__((always_inline)) {
                u32x4 r;
                asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(xa + rd[ks]), "i"(4096 * decltype(I)::value));
                fa[decltype(I)::value] = r;
            });
            // the other buffer was last read in phase 3 of step s - 1; every wave's reads of that phase were complete
            // before the barrier that ended it (lgkmcnt(0) below)
            if (s + 1 < nk) {
                if constexpr (ks == 0) issue(s + 1, I0{}, IH{});
                if constexpr (ks == 1) issue(s + 1, IH{}, IE{});
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            // the next step's loads are complete before the barrier after which waves 0 .. 3 read them: for waves 4 .. 7
            // that is this one, for waves 0 .. 3 the one that ends the phase
            if constexpr (ks == 3) {
                if (behind) __builtin_amdgcn_s_waitcnt(0x0F70);
            }
            barrier();
            if (!HALF || ks < 2 || s + 1 < nk) {
#pragma unroll
                for (int i = 0; i < kBigMI; i++)
#pragma unroll
                    for (int j = 0; j < kBigNJ; j++) acc[i][j] = mfma32x32x16(as_half8(fa[i]), as_half8(fb[j]), acc[i][j]);
            }
            if constexpr (ks == 3) {
                if (!behind) __builtin_amdgcn_s_waitcnt(0x0F70);
            }
            barrier();
        });
    }
    if (!behind) barrier();  // the barrier that the other half began with

    // lane holds Y[m0 + (256 / WM) wm + 32 i + 8 (v / 4) + 4 hi + v % 4][n0 + WC wn + 32 j + l32]
#pragma unroll
    for (int i = 0; i < kBigMI; i++)
#pragma unroll
        for (int j = 0; j < kBigNJ; j++) {
            const int n = n0 + WC * wn + 32 * j + l32;
            if (n < p.N) store_col16<OUT16>(p, mi, n, m0 + (kBM / WM) * wm + 32 * i + 4 * hi, acc[i][j]);
        }
}

template <bool OUT16, bool HALF>
__global__ __launch_bounds__(kBigThreads, 1) void gemm_big_kernel(LinearParams p) { gemm_big_tile<OUT16, 256, 64, HALF>(p); }
template <bool OUT16, bool HALF>
__global__ __launch_bounds__(kBigThreads, 1) void gemm_w192_kernel(LinearParams p) { gemm_big_tile<OUT16, 192, 96, HALF>(p); }

// ---- M > 8, products with too few 256-row tiles for the chip: BM x BN tiles of 4 waves, K cut into p.plan.splits parts
// Few rows are bound by the weights' stream from HBM (24 x 4096 x 4096: 33.5 MB, 5.2 us at 6.4 TB/s), which needs every
// CU loading: with whole K a product of N = 4096 has 32 column tiles for 256 CUs, so the parts of K make up the rest
// (4 parts of 64-column tiles: 256 workgroups). Each workgroup keeps NBUF - 1 steps of both operands in flight straight
// into LDS (32 to 100 KB), in whole row slices of 256 (BK = 128) or 128 bytes, so its few steps arrive about together.
// Row r of a tile lies whole in LDS with its 16-byte chunks permuted by the row (chunk ^ r % 16, or ^ r / 2 % 8 with
// 128-byte rows): the 16-byte operand reads of 16 rows at one chunk hit 16 distinct 4-bank groups. The weights are MFMA
// operand A, so that a lane holds 4 consecutive outputs of one row (16-byte stores).
// HALF: K is an odd multiple of 32, as in gemm_big_tile; the last part's last step is half padding. WIDE: the tile's rows
// span 4 GiB or more, so the lanes' offsets take 64 bits.
template <bool OUT16, int BM, int BN, int WM, int BK, int NBUF, bool HALF, bool WIDE>
__device__ __forceinline__ void gemm_split_tile(const LinearParams & p) {
    constexpr int WN = kWaves / WM;                        // waves along the weight rows
    constexpr int MI = BM / WM / 16, NJ = BN / WN / 16;    // 16 x 16 MFMA tiles per wave
    constexpr int RPB = 512 / BK;                          // rows per 1 KB load block
    constexpr int XB = BM / RPB, WB = BN / RPB;            // load blocks of a step
    constexpr int LPS = (XB + WB) / kWaves;                // loads per wave and step
    constexpr int KS = BK / 32;                            // MFMA steps per K step
    static_assert(!HALF || BK == 64, "a last step of 32 columns and 32 of padding");
    static_assert((XB + WB) % kWaves == 0 && MI >= 1 && NJ >= 1 && LPS * (NBUF - 1) < 64, "whole loads and tiles");
    __shared__ __attribute__((aligned(1024))) half_t sm[NBUF][(BM + BN) * BK];
    __shared__ int s_last;
    const int n_tiles = (p.N + BN - 1) / BN, m_tiles = (p.M + BM - 1) / BM, S = p.plan.splits;
    uint32_t t = xcd_remap(blockIdx.x, (uint32_t)(p.plan.tiles * S));
    const int mt = t % m_tiles;
    t /= m_tiles;
    const int split = t % S;
    t /= S;
    const int nt = t % n_tiles, mi = t / n_tiles;
    const int tile = (mi * n_tiles + nt) * m_tiles + mt;
    const int m0 = mt * BM, n0 = nt * BN;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    const int kp = HALF ? p.K + 32 : p.K;
    const int steps = kp / BK, s0 = (int)((int64_t)split * steps / S), nk = (int)((int64_t)(split + 1) * steps / S) - s0;

    // load block i kWaves + wave of a step (see gemm_block_row)
    const char * const xg = reinterpret_cast<const char *>(p.xh + (int64_t)m0 * kp);
    const char * const wg = reinterpret_cast<const char *>(p.w[mi] + (int64_t)n0 * p.K);
    using Offset = std::conditional_t<WIDE, uint64_t, uint32_t>;
    Offset off[LPS];
#pragma unroll
    for (int i = 0; i < LPS; i++) {
        const int j = i * kWaves + wave, jb = j < XB ? j : j - XB;
        const int row = gemm_block_row<BK>(jb, lane), chunk = gemm_block_chunk<BK>(jb, lane);
        off[i] = j < XB ? gemm_load_offset<Offset>(m0, row, p.M, kp, chunk)
                        : gemm_load_offset<Offset>(n0, row, p.N, p.K, chunk);
    }
    auto issue = [&](int step, int buf) __attribute__((always_inline)) {
        const int64_t k0 = (int64_t)(s0 + step) * BK * 2;
        const bool half_step = HALF && (s0 + step) * BK + BK > p.K;
#pragma unroll
        for (int i = 0; i < LPS; i++) {
            const int j = i * kWaves + wave;
            const char * src = (j < XB ? xg : wg) + k0;
            Offset o = off[i];
            if (half_step && j >= XB) o -= gemm_half_back(gemm_block_chunk<BK>(j - XB, lane));
            __builtin_amdgcn_global_load_lds(src + o, (__attribute__((address_space(3))) void *)&sm[buf][512 * j], 16, 0, 0);
        }
    };
    float4_t acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
    const int wm = wave / WN, wn = wave % WN, l16 = lane % 16, grp = lane / 16;
    uint32_t rd[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) rd[ks] = (uint32_t)l16 * BK * 2 + 16 * ((4 * ks + grp) ^ gemm_swizzle<BK>(l16));
    const uint32_t lds0 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) half_t *)sm[0];
#pragma unroll
    for (int a = 0; a < NBUF - 1; a++)
        if (a < nk) issue(a, a);
    for (int s = 0; s < nk; s++) {
        const int buf = s % NBUF;
        const bool half_step = HALF && (s0 + s) * BK + BK > p.K;
        const int later = min(NBUF - 2, nk - 1 - s);
        static_for<0, NBUF - 1>([&](auto R) __attribute__((always_inline)) {
            constexpr int n = decltype(R)::value * LPS;
            if (later == decltype(R)::value) __builtin_amdgcn_s_waitcnt(0x0F70 | (n & 15) | ((n >> 4) << 14));
        });
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (s + NBUF - 1 < nk) issue(s + NBUF - 1, (s + NBUF - 1) % NBUF);
        const uint32_t xa = lds0 + (uint32_t)buf * (BM + BN) * BK * 2 + wm * (BM / WM) * BK * 2;
        const uint32_t wa = lds0 + (uint32_t)buf * (BM + BN) * BK * 2 + (BM + wn * (BN / WN)) * BK * 2;
        u32x4 fx[KS][MI], fw[KS][NJ];
        auto reads = [&](auto KSC) __attribute__((always_inline)) {
            constexpr int ks = decltype(KSC)::value;
            static_for<0, MI>([&](auto I) __attribute__((always_inline)) {
                u32x4 r;
                asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(xa + rd[ks]), "i"(32 * BK * decltype(I)::value));
                fx[ks][decltype(I)::value] = r;
            });
            static_for<0, NJ>([&](auto J) __attribute__((always_inline)) {
                u32x4 r;
                asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(wa + rd[ks]), "i"(32 * BK * decltype(J)::value));
                fw[ks][decltype(J)::value] = r;
            });
        };
        reads(std::integral_constant<int, 0>{});
        reads(std::integral_constant<int, 1>{});
        static_for<0, KS>([&](auto KSC) __attribute__((always_inline)) {
            constexpr int ks = decltype(KSC)::value;
            if constexpr (ks + 1 < KS) asm volatile("s_waitcnt lgkmcnt(%0)" ::"i"(MI + NJ) : "memory");
            else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            if (!HALF || ks == 0 || !half_step) {
#pragma unroll
                for (int i = 0; i < MI; i++)
#pragma unroll
                    for (int j = 0; j < NJ; j++) acc[i][j] = mfma16x16x32(as_half8(fw[ks][j]), as_half8(fx[ks][i]), acc[i][j]);
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (ks + 2 < KS) reads(std::integral_constant<int, ks + 2>{});
        });
    }

    if (S > 1) {
        // the partial tile out with device-scope stores, complete before the tile's counter counts it in; the part that
        // completes the count sums every part in order (its own read back too: the result does not depend on which part
        // came last) and writes the output
        constexpr int64_t TF = (int64_t)BM * BN;  // floats per partial tile
        const __amdgpu_buffer_rsrc_t prs = dev_rsrc(p.part + (int64_t)tile * S * TF);
        const int fb = ((wave * MI * NJ) * kWave + lane) * 16;
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++) store16_dev(prs, split * (int)TF * 4 + fb + (i * NJ + j) * kWave * 16, acc[i][j]);
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (threadIdx.x == 0)
            s_last = __hip_atomic_fetch_add(p.counters + (int64_t)tile * kCounterStride, 1u, __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT) == (uint32_t)(S - 1);
        __syncthreads();
        if (!s_last) return;
        __builtin_amdgcn_s_waitcnt(0);
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
        constexpr int SC = MI * NJ >= 16 ? 1 : 16 / (MI * NJ);  // parts in flight per round
        for (int k0 = 0; k0 < S; k0 += SC) {
            float4_t v[SC][MI][NJ];
#pragma unroll
            for (int e = 0; e < SC; e++)
                if (k0 + e < S)
#pragma unroll
                    for (int i = 0; i < MI; i++)
#pragma unroll
                        for (int j = 0; j < NJ; j++)
                            v[e][i][j] = __builtin_bit_cast(
                                float4_t, load16_dev(prs, (k0 + e) * (int)TF * 4 + fb + (i * NJ + j) * kWave * 16));
#pragma unroll
            for (int e = 0; e < SC; e++)
                if (k0 + e < S)
#pragma unroll
                    for (int i = 0; i < MI; i++)
#pragma unroll
                        for (int j = 0; j < NJ; j++) acc[i][j] += v[e][i][j];
        }
    }

    // lane holds Y[m0 + wm BM / WM + 16 i + l16][n0 + wn BN / WN + 16 j + 4 grp + v]
    const float * b = (p.flags & kLinearBias) ? p.bias[mi] : nullptr;
    const bool accum = p.flags & kLinearAccumulate;
    const int mb = m0 + wm * (BM / WM) + l16, nb = n0 + wn * (BN / WN) + 4 * grp;
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const int n = nb + 16 * j;
        if (n >= p.N) continue;
        const bool whole = n + 3 < p.N;
        if (b) {
            float bv[4];
#pragma unroll
            for (int v = 0; v < 4; v++) bv[v] = b[min(n + v, p.N - 1)];
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int v = 0; v < 4; v++) acc[i][j][v] += bv[v];
        }
        if (accum) {
            float prev[MI][4];
#pragma unroll
            for (int i = 0; i < MI; i++) {
                const int64_t o = (int64_t)min(mb + 16 * i, p.M - 1) * p.y_stride + n;
#pragma unroll
                for (int v = 0; v < 4; v++) prev[i][v] = 0.f;
                if (whole) {
                    if constexpr (OUT16) {
                        const half4_t h = *reinterpret_cast<const half4_t *>(static_cast<const half_t *>(p.y[mi]) + o);
#pragma unroll
                        for (int v = 0; v < 4; v++) prev[i][v] = (float)h[v];
                    } else {
                        const float4_t h = *reinterpret_cast<const float4_t *>(static_cast<const float *>(p.y[mi]) + o);
#pragma unroll
                        for (int v = 0; v < 4; v++) prev[i][v] = h[v];
                    }
                } else {
#pragma unroll
                    for (int v = 0; v < 4; v++)
                        if (n + v < p.N)
                            prev[i][v] = OUT16 ? (float)static_cast<const half_t *>(p.y[mi])[o + v]
                                               : static_cast<const float *>(p.y[mi])[o + v];
                }
            }
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int v = 0; v < 4; v++) acc[i][j][v] += prev[i][v];
        }
#pragma unroll
        for (int i = 0; i < MI; i++) {
            const int m = mb + 16 * i;
            if (m >= p.M) continue;
            const int64_t o = (int64_t)m * p.y_stride + n;
            if constexpr (OUT16) {
                half_t * y = static_cast<half_t *>(p.y[mi]) + o;
                const float4_t a = acc[i][j];
                if (whole) *reinterpret_cast<half4_t *>(y) = half4_t{(half_t)a[0], (half_t)a[1], (half_t)a[2], (half_t)a[3]};
                else
#pragma unroll
                    for (int v = 0; v < 3; v++)
                        if (n + v < p.N) y[v] = (half_t)acc[i][j][v];
            } else {
                float * y = static_cast<float *>(p.y[mi]) + o;
                if (whole) *reinterpret_cast<float4_t *>(y) = acc[i][j];
                else
#pragma unroll
                    for (int v = 0; v < 3; v++)
                        if (n + v < p.N) y[v] = acc[i][j][v];
            }
        }
    }
}

template <bool OUT16, int BM, int BN, int WM, int BK, int NBUF, bool HALF, bool WIDE>
__global__ __launch_bounds__(kThreads, 1) void gemm_split_kernel(LinearParams p) {
    gemm_split_tile<OUT16, BM, BN, WM, BK, NBUF, HALF, WIDE>(p);
}

// The kernels of kGemmCfgs, by shape: f32 and f16 outputs, and those of a K that is an odd multiple of 32, for the shapes
// that take one.
struct GemmKernels {
    int threads;
    void (*k32)(LinearParams);
    void (*k16)(LinearParams);
    void (*half32)(LinearParams);
    void (*half16)(LinearParams);
};
template <int BM, int BN, int WM, int BK, int NBUF, bool WIDE = false>
constexpr GemmKernels split_kernels() {
    GemmKernels k{kThreads, gemm_split_kernel<false, BM, BN, WM, BK, NBUF, false, WIDE>,
                  gemm_split_kernel<true, BM, BN, WM, BK, NBUF, false, WIDE>, nullptr, nullptr};
    if constexpr (BK == 64) {
        k.half32 = gemm_split_kernel<false, BM, BN, WM, BK, NBUF, true, WIDE>;
        k.half16 = gemm_split_kernel<true, BM, BN, WM, BK, NBUF, true, WIDE>;
    }
    return k;
}
const GemmKernels & gemm_kernels(int cfg) {
    static const GemmKernels kernels[kNumGemmCfgs] = {
        split_kernels<16, 64, 1, 128, 6>(),
        split_kernels<32, 64, 1, 128, 3>(),
        split_kernels<64, 64, 2, 64, 4>(),
        split_kernels<128, 64, 2, 128, 3>(),
        split_kernels<128, 128, 2, 64, 4>(),
        split_kernels<128, 128, 2, 64, 2>(),
        {kBigThreads, gemm_w192_kernel<false, false>, gemm_w192_kernel<true, false>, gemm_w192_kernel<false, true>,
         gemm_w192_kernel<true, true>},
        {kBigThreads, gemm_big_kernel<false, false>, gemm_big_kernel<true, false>, gemm_big_kernel<false, true>,
         gemm_big_kernel<true, true>},
        split_kernels<64, 64, 2, 64, 4, true>(),
    };
    return kernels[cfg];
}

// Waves per workgroup: the (matrix, RW-row group) items spread evenly over the CUs, one workgroup per CU (the weight
// stream of each CU then ends at the same time), up to 8 waves; beyond 2048 items, several workgroups of 8 per CU.
template <int MT, int RW>
hipError_t launch_gemv_rw(const LinearParams & p, hipStream_t stream) {
    const int64_t items = (int64_t)((p.N + RW - 1) / RW) * p.count;
    const int nw = (int)std::min<int64_t>(kGemvMaxWaves, std::max<int64_t>(1, (items + 255) / 256));
    const dim3 grid((uint32_t)((items + nw - 1) / nw));
    const dim3 block((uint32_t)(nw * kWave));
    const size_t lds = (size_t)MT * p.K * sizeof(float);
    const int v = (lds <= kLinearGemvLds ? 4 : 0) | ((p.flags & kLinearOutF16) ? 2 : 0) | ((p.flags & kLinearNorm) ? 1 : 0);
    const size_t dyn = (v & 4) ? lds : 0;
    switch (v) {
        case 0: hipLaunchKernelGGL((gemv_kernel<MT, false, false, false, RW>), grid, block, dyn, stream, p); break;
        case 1: hipLaunchKernelGGL((gemv_kernel<MT, false, false, true, RW>), grid, block, dyn, stream, p); break;
        case 2: hipLaunchKernelGGL((gemv_kernel<MT, false, true, false, RW>), grid, block, dyn, stream, p); break;
        case 3: hipLaunchKernelGGL((gemv_kernel<MT, false, true, true, RW>), grid, block, dyn, stream, p); break;
        case 4: hipLaunchKernelGGL((gemv_kernel<MT, true, false, false, RW>), grid, block, dyn, stream, p); break;
        case 5: hipLaunchKernelGGL((gemv_kernel<MT, true, false, true, RW>), grid, block, dyn, stream, p); break;
        case 6: hipLaunchKernelGGL((gemv_kernel<MT, true, true, false, RW>), grid, block, dyn, stream, p); break;
        default: hipLaunchKernelGGL((gemv_kernel<MT, true, true, true, RW>), grid, block, dyn, stream, p); break;
    }
    return hipGetLastError();
}

// Rows per wave: 2 where the items still fit one workgroup per CU, i.e. twice the waves streaming the same bytes
// (A/B on one box, us per launch: Llama-3-8B attention output 8.77 -> 8.41, a 14336-column down projection
// 23.36 -> 22.69, Whisper attention output 3.73 -> 3.63, Qwen2.5-0.5B 3.33 -> 3.24, eight input rows 21.2 -> 19.7;
// unchanged at two rows and the q|k|v width, which takes 4 rows per wave to fit). Four input rows keep 4 rows per
// wave: with 2 they ran 16.5 -> 20.2 us.
template <int MT>
hipError_t launch_gemv_t(const LinearParams & p, hipStream_t stream) {
    const int64_t cap = (int64_t)256 * kGemvMaxWaves;  // one workgroup of at most 8 waves per CU
    if (MT != 4 && (int64_t)((p.N + 1) / 2) * p.count <= cap) return launch_gemv_rw<MT, 2>(p, stream);
    return launch_gemv_rw<MT, kGemvRows>(p, stream);
}

}  // namespace

hipError_t launch_stage(const LinearParams & p, hipStream_t stream) {
    if (p.flags & kLinearNorm) hipLaunchKernelGGL(stage_kernel<true>, dim3((uint32_t)p.M), dim3(kThreads), 0, stream, p);
    else hipLaunchKernelGGL(stage_kernel<false>, dim3((uint32_t)p.M), dim3(kThreads), 0, stream, p);
    return hipGetLastError();
}

hipError_t launch_linear(const LinearParams & p, hipStream_t stream) {
    if (p.M <= kLinearGemvMaxRows) {
        if (p.M <= 1) return launch_gemv_t<1>(p, stream);
        if (p.M <= 2) return launch_gemv_t<2>(p, stream);
        if (p.M <= 4) return launch_gemv_t<4>(p, stream);
        return launch_gemv_t<8>(p, stream);
    }
    if (hipError_t e = launch_stage(p, stream); e != hipSuccess) return e;
    return launch_gemm(p, stream);
}

hipError_t launch_gemm(const LinearParams & p, hipStream_t stream) {
    const GemmKernels & k = gemm_kernels(p.plan.cfg);
    const bool out16 = p.flags & kLinearOutF16, half = p.K % 64 != 0;
    hipLaunchKernelGGL(half ? (out16 ? k.half16 : k.half32) : (out16 ? k.k16 : k.k32), dim3((uint32_t)(p.plan.tiles * p.plan.splits)),
                       dim3(k.threads), 0, stream, p);
    return hipGetLastError();
}

}  // namespace mx
