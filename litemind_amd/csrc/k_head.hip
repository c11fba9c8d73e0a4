// k_head.hip -- the LM head and the greedy choice of the next token.
//
// Reference: the end of DeepSeekRunner::Impl::forward (src/DeepSeekRunner.cpp:
// 296-300): rms_norm with the final norm weight, then gemm::matvec_bf16 over
// the [V, H] head; and Sampler::select_next's greedy branch
// (src/Sampler.cpp:117-126), std::max_element over the logits.
//
// The logits follow gemm::dot_bf16's association (src/Gemm.cpp:46-82) bit for
// bit, like gemv_plain_kernel: 32 sequential fused chains over the elements
// i = c (mod 32), chains 0..7 continuing over the 8-wide remainder, then
// (a0+a1)+(a2+a3) per lane, lanes j and j+4 added, (h0+h2)+(h1+h3) (no scalar
// tail: the width is a multiple of 8).  A chain's elements lie 64 bytes apart;
// a lane that owns 8 consecutive chains reads one 16-byte piece per step, so
// the loads stay wide and every chain stays in one lane, in order.  The head
// streams 420 MB at V = 102400, H = 2048: the kernel is bound by HBM.
#include "lm_internal.h"

#include <algorithm>

namespace lm {
namespace {

constexpr int kThreads = 256;                            // the head: 4 waves per block
constexpr int kRowsPerWave = 16;                         // 4 lanes per row
constexpr int kRows = kRowsPerWave * (kThreads / 64);    // head rows per block
constexpr int kUnroll = 8;                               // 16-byte loads in flight per lane
// Projections with few rows (attention: 576 to 4096) take one wave per block,
// so that a launch still spreads over the CUs.
constexpr int kSmallThreads = 64;

// Combines two candidates of the greedy choice: the larger value, the lower
// index between equal values (IEEE equality: -0 equals +0), NaN never chosen.
// Associative, so the order of the reduction does not matter.
__device__ inline HeadBest better(HeadBest a, HeadBest b) {
    if (!b.have) {
        return a;
    }
    if (!a.have || b.v > a.v || (b.v == a.v && b.i < a.i)) {
        return b;
    }
    return a;
}

// Row `row`'s candidate.  A NaN is none, except at index 0, which nothing after
// it can replace: the largest value at the lowest index.
__device__ inline HeadBest candidate(float logit, int64_t row, bool live) {
    const bool nan = logit != logit;
    return {nan && row == 0 ? __builtin_inff() : logit, static_cast<int32_t>(row), live && (!nan || row == 0) ? 1 : 0};
}

__device__ inline HeadBest wave_better(HeadBest b) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const HeadBest other{__shfl_xor(b.v, o), __shfl_xor(b.i, o), __shfl_xor(b.have, o)};
        b = better(b, other);
    }
    return b;
}

// Four lanes per row: lane q of a row owns chains 8q .. 8q + 7, so one 16-byte
// load gives it the next element of each of its chains (elements 32 s + 8 q ..
// + 7), and a wave's load covers 64 contiguous bytes of 16 rows.  The tokens
// (tokens x in_dim floats, dynamic LDS) are staged once per block.  Lane 0 of a
// row also owns chains 0..7's continuation over the 8-wide remainder.  Then
// each block's best row per token goes to `partial` (when given; `logits` may
// then be null: a [102400] head kept 26 MB for the logits of 64 tokens that a
// caller did not ask for).
template <int THREADS>
__global__ __launch_bounds__(THREADS) void head_logits_kernel(const uint16_t* __restrict__ w,
                                                              const float* __restrict__ x, float* logits,
                                                              HeadBest* partial, int64_t rows, int32_t in_dim,
                                                              int32_t tokens, float scale, int32_t accumulate) {
    constexpr int ROWS = kRowsPerWave * (THREADS / 64);
    extern __shared__ float4 xs4[];  // [tokens][in_dim / 4]
    __shared__ HeadBest wave_best[THREADS / 64];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int q = lane & 3;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * ROWS + (tid >> 2);
    const bool live = row < rows;
    const int n32 = in_dim / 32 * 32;
    const int n8 = n32 + (in_dim - n32) / 8 * 8;  // == in_dim: the launch requires in_dim % 8 == 0
    const int q4 = in_dim / 4;
    const float4* x4 = reinterpret_cast<const float4*>(x);
    for (int i = tid; i < tokens * q4; i += THREADS) {
        xs4[i] = x4[i];
    }
    __syncthreads();
    const uint16_t* wr = w + (live ? row : rows - 1) * in_dim;
    float acc[kHeadTokens][8];
#pragma unroll
    for (int t = 0; t < kHeadTokens; ++t) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            acc[t][j] = 0.0f;
        }
    }
    auto step = [&](const uint4 wv, int e) {
        // elements e .. e + 7 of the row, chains (e % 32) .. + 7
        float wf[8];
        wf[0] = widen_bf16(static_cast<uint16_t>(wv.x));
        wf[1] = widen_bf16(static_cast<uint16_t>(wv.x >> 16));
        wf[2] = widen_bf16(static_cast<uint16_t>(wv.y));
        wf[3] = widen_bf16(static_cast<uint16_t>(wv.y >> 16));
        wf[4] = widen_bf16(static_cast<uint16_t>(wv.z));
        wf[5] = widen_bf16(static_cast<uint16_t>(wv.z >> 16));
        wf[6] = widen_bf16(static_cast<uint16_t>(wv.w));
        wf[7] = widen_bf16(static_cast<uint16_t>(wv.w >> 16));
#pragma unroll
        for (int t = 0; t < kHeadTokens; ++t) {
            if (t < tokens) {
                const float4 xa = xs4[t * q4 + e / 4];
                const float4 xb = xs4[t * q4 + e / 4 + 1];
                acc[t][0] = __builtin_fmaf(wf[0], xa.x, acc[t][0]);
                acc[t][1] = __builtin_fmaf(wf[1], xa.y, acc[t][1]);
                acc[t][2] = __builtin_fmaf(wf[2], xa.z, acc[t][2]);
                acc[t][3] = __builtin_fmaf(wf[3], xa.w, acc[t][3]);
                acc[t][4] = __builtin_fmaf(wf[4], xb.x, acc[t][4]);
                acc[t][5] = __builtin_fmaf(wf[5], xb.y, acc[t][5]);
                acc[t][6] = __builtin_fmaf(wf[6], xb.z, acc[t][6]);
                acc[t][7] = __builtin_fmaf(wf[7], xb.w, acc[t][7]);
            }
        }
    };
    const int steps = n32 / 32;
    int s = 0;
    for (; s + kUnroll <= steps; s += kUnroll) {
        uint4 wv[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            wv[u] = load_stream16(wr + 32 * (s + u) + 8 * q);
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            step(wv[u], 32 * (s + u) + 8 * q);
        }
    }
    for (; s < steps; ++s) {
        step(load_stream16(wr + 32 * s + 8 * q), 32 * s + 8 * q);
    }
    if (q == 0) {
        // chains 0..7 continue over the remainder, element n32 + 8 k + j on chain j
        for (int e = n32; e < n8; e += 8) {
            step(load_stream16(wr + e), e);
        }
    }
#pragma unroll
    for (int t = 0; t < kHeadTokens; ++t) {
        if (t >= tokens) {
            break;
        }
        // lane sums (a[l] + a[8 + l]) + (a[16 + l] + a[24 + l]) over the row's 4 lanes
        float ls[8];
#pragma unroll
        for (int l = 0; l < 8; ++l) {
            const float v01 = acc[t][l] + __shfl_xor(acc[t][l], 1);
            ls[l] = v01 + __shfl_xor(v01, 2);
        }
        const float h0 = ls[0] + ls[4];
        const float h1 = ls[1] + ls[5];
        const float h2 = ls[2] + ls[6];
        const float h3 = ls[3] + ls[7];
        const float total = (h0 + h2) + (h1 + h3);
        if (live && q == 0 && logits != nullptr) {
            // gemm::matvec_bf16_accumulate folds the row as fma(scale, dot, out) (src/Gemm.cpp:156-175)
            float* o = logits + static_cast<int64_t>(t) * rows + row;
            *o = accumulate ? __builtin_fmaf(scale, total, *o) : total;
        }
        if (partial == nullptr) {
            continue;
        }
        HeadBest b = candidate(total, row, live && q == 0);
        b = wave_better(b);
        if (lane == 0) {
            wave_best[tid >> 6] = b;
        }
        __syncthreads();
        if (tid == 0) {
            HeadBest r = wave_best[0];
            for (int k = 1; k < THREADS / 64; ++k) {
                r = better(r, wave_best[k]);
            }
            partial[static_cast<int64_t>(t) * gridDim.x + blockIdx.x] = r;
        }
        __syncthreads();
    }
}

// ---- the same dot products for batches of tokens, on the fp32 matrix cores ----
//
// v_mfma_f32_*_f32 forms each output as a chain of fused multiply-adds over k
// in ascending order, each rounded as fmaf rounds it, subnormals included
// (checked bit for bit against fmaf on the host over normal, subnormal,
// overflowing and signed-zero operands for the 32x32x2 and 16x16x4 shapes).
// dot_bf16's 32 chains are chains of exactly that kind, so one accumulator
// tile per chain gives every (token, row) pair's chain bit for bit: the k
// index of one instruction runs over the 2 (or 4) successive 32-element steps
// of the row, and its operands are one chain's elements of those steps.
//
// A workgroup's four waves own 8 chains each (chains 8 w .. 8 w + 7) of one
// tile of tokens x rows, so a chain's whole sum stays in one register and the
// four waves share every staged byte.  Tiles: 32 tokens x 32 rows
// (32x32x2, 128 accumulators per lane), or 16 tokens x 16 NR rows (16x16x4).
// A stage is 64 (or 128) elements of the tile's rows and tokens, loaded
// straight to LDS with its 16-byte units XOR-swizzled by row against bank
// conflicts; DEPTH stages are in flight.  Each wave reads the next stage's operands before this
// stage's MFMAs, which hide the reads.  At the end the waves exchange their
// chains through the ring's LDS and reduce them in dot_bf16's order.
//
// What bounds it: the fp32 matrix rate (134 TFLOP/s measured for 32x32x2) at
// 32 and more tokens, the weight stream below.  [102400, 2048] head, launches in
// a row: 16 tokens 106 us (4.0 TB/s), 32 tokens 155 us (87 TFLOP/s); whole calls
// 116 and 166 us, 416 and 833 with the few-token kernel's launches of 4.  [3072,
// 2048] projection of 77 tokens 15 us (VALU chains, one token per lane: about
// 35).  Small projections end with their longest wave: 16 stages of 8 chains.
// s_waitcnt immediate: vmcnt(n) (bits 3:0 and 15:14), the other counters unconstrained
constexpr int kWaitVm(int n) { return (n & 15) | ((n >> 4) << 14) | 0x0070 | 0x0F00; }

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// One chain's accumulator over the wave's tile: M tokens x (M NR) rows.
template <int M, int NR>
struct ChainTile;
template <int NR>
struct ChainTile<32, NR> {
    static_assert(NR == 1);
    f32x16 v = {};
    __device__ void step(const float* a, const float (*b)[8], int j) {
        v = __builtin_amdgcn_mfma_f32_32x32x2f32(a[j], b[0][j], v, 0, 0, 0);
    }
    __device__ float get(int quarter, int i) const { return v[4 * quarter + i]; }
};
template <int NR>
struct ChainTile<16, NR> {
    f32x4 v[NR] = {};
    __device__ void step(const float* a, const float (*b)[8], int j) {
#pragma unroll
        for (int n = 0; n < NR; ++n) {
            v[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[n][j], v[n], 0, 0, 0);
        }
    }
    __device__ float get(int quarter, int i) const { return v[i][quarter]; }
};

template <int M, int NR>
struct ExactTile {
    static constexpr int kSteps = M == 32 ? 2 : 4;       // 32-element steps per instruction and stage
    static constexpr int kElems = 32 * kSteps;           // row elements per stage
    static constexpr int kRowsT = M * NR;                // weight rows per tile
    static constexpr int kXUnits = kElems / 4;           // 16-byte units of a token's stage
    static constexpr int kWUnits = kElems / 8;           // 16-byte units of a row's stage
    static constexpr int kXLoads = M * kXUnits / 256;    // loads per wave and stage
    static constexpr int kWLoads = kRowsT * kWUnits / 256;
    static constexpr int kLoads = kXLoads + kWLoads;
    static constexpr int kStageFloats = M * kElems + kRowsT * kElems / 2;
    static constexpr int kQuarter = M == 32 ? 4 : NR;    // accumulators of a chain that one wave finishes
    static_assert(kXLoads >= 1 && kWLoads >= 1);
    // A 16-byte LDS read serves 16 lanes: 16 successive rows take 16 different
    // columns of banks (rows of 128 bytes alternate between two halves).
    static __device__ int wswizzle(int r) { return kWUnits == 8 ? (r >> 1) & 7 : r & 15; }
};

// in_dim % (32 kSteps) == 0.  `nt` token tiles, `nr` row tiles; workgroups that
// share rows lie 8 apart in the grid, on one XCD.
template <int M, int NR, int DEPTH, bool BEST>
__global__ __launch_bounds__(256, 2) void matvec_exact_kernel(const uint16_t* __restrict__ w,
                                                              const float* __restrict__ x, float* out,
                                                              HeadBest* partial, int64_t rows, int32_t in_dim,
                                                              int32_t tokens, int32_t nt, int32_t nr, float scale,
                                                              int32_t accumulate) {
    using T = ExactTile<M, NR>;
    // One array per stage, so that the compiler's waits tell the stages apart.
    __shared__ __align__(16) float s0[T::kStageFloats], s1[T::kStageFloats], s2[T::kStageFloats],
        s3[T::kStageFloats], s4[DEPTH > 4 ? T::kStageFloats : 1], s5[DEPTH > 5 ? T::kStageFloats : 1];
    static_assert(DEPTH >= 4 && DEPTH <= 6);
    float* const ring[6] = {s0, s1, s2, s3, s4, s5};
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int slot_id = static_cast<int>(blockIdx.x) / 8;
    const int tt = slot_id % nt;
    const int rt = slot_id / nt * 8 + static_cast<int>(blockIdx.x) % 8;
    if (rt >= nr) {
        return;
    }
    const int t0 = tt * M;
    const int ntok = min(M, tokens - t0);
    const int64_t row0 = static_cast<int64_t>(rt) * T::kRowsT;
    const int nrow = static_cast<int>(std::min<int64_t>(T::kRowsT, rows - row0));
    const int stages = in_dim / T::kElems;
    const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(x + static_cast<int64_t>(t0) * in_dim), 0, ntok * in_dim * 4, kBufferWord3);
    const __amdgpu_buffer_rsrc_t wres =
        __builtin_amdgcn_make_buffer_rsrc((void*)(w + row0 * in_dim), 0, nrow * in_dim * 2, kBufferWord3);
    // Load j of a stage fills 64 consecutive 16-byte positions p; position p of
    // token r = p / units holds its unit (p % units) ^ (r % 16), of a weight row
    // (p % units) ^ wswizzle(r).  Rows past the end load the last one.
    unsigned xsrc[T::kXLoads], wsrc[T::kWLoads];
#pragma unroll
    for (int j = 0; j < T::kXLoads; ++j) {
        const int p = (wave * T::kXLoads + j) * 64 + lane;
        const int r = p / T::kXUnits;
        const int u = (p % T::kXUnits) ^ (r & 15);
        xsrc[j] = static_cast<unsigned>((min(r, ntok - 1) * in_dim + 4 * u) * 4);
    }
#pragma unroll
    for (int j = 0; j < T::kWLoads; ++j) {
        const int p = (wave * T::kWLoads + j) * 64 + lane;
        const int r = p / T::kWUnits;
        const int u = (p % T::kWUnits) ^ T::wswizzle(r);
        wsrc[j] = static_cast<unsigned>((min(r, nrow - 1) * in_dim + 8 * u) * 2);
    }
    auto issue = [&](int stage, float* slot) {
        stage = stage < stages ? stage : stages - 1;  // past the end: the last again (every stage issues alike)
#pragma unroll
        for (int j = 0; j < T::kXLoads; ++j) {
            buffer_lds16(xres, slot + (wave * T::kXLoads + j) * 256, xsrc[j], stage * (T::kElems * 4));
        }
#pragma unroll
        for (int j = 0; j < T::kWLoads; ++j) {
            buffer_lds16(wres, slot + M * T::kElems + (wave * T::kWLoads + j) * 256, wsrc[j], stage * (T::kElems * 2));
        }
    };
    // This lane's operands of a stage: step k = lane / M of token and row
    // lane % M, the wave's 8 chains.
    const int li = lane % M;
    const int lk = lane / M;
    const int xu = 8 * lk + 2 * wave;
    const int wu = 4 * lk + wave;
    auto read = [&](const float* slot, f32x4 (&xv)[2], uint4 (&wv)[NR]) {
        xv[0] = *reinterpret_cast<const f32x4*>(slot + li * T::kElems + 4 * (xu ^ (li & 15)));
        xv[1] = *reinterpret_cast<const f32x4*>(slot + li * T::kElems + 4 * ((xu + 1) ^ (li & 15)));
#pragma unroll
        for (int n = 0; n < NR; ++n) {
            const int r = n * M + li;
            wv[n] = *reinterpret_cast<const uint4*>(slot + M * T::kElems + r * (T::kElems / 2) +
                                                    4 * (wu ^ T::wswizzle(r)));
        }
    };
    ChainTile<M, NR> acc[8];
    auto mfma = [&](const f32x4 (&xv)[2], const uint4 (&wv)[NR]) {
        float a[8], b[NR][8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            a[j] = xv[j / 4][j % 4];
        }
#pragma unroll
        for (int n = 0; n < NR; ++n) {
            const uint32_t pair[4] = {wv[n].x, wv[n].y, wv[n].z, wv[n].w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                b[n][2 * j] = bits_float(pair[j] << 16);
                b[n][2 * j + 1] = bits_float(pair[j] & 0xffff0000u);
            }
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            acc[j].step(a, b, j);
        }
    };
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d) {
        issue(d, ring[d]);
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(kWaitVm(T::kLoads * (DEPTH - 2)));  // stage 0 is in
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    f32x4 xv[2][2];
    uint4 wv[2][NR];
    read(ring[0], xv[0], wv[0]);
    auto stage_step = [&](int s, int u) {  // u: s modulo kTrip, a constant once unrolled
        // stage s + 1 is in, and every wave has the operands of s - 1: its slot
        // takes stage s + DEPTH - 1
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(kWaitVm(T::kLoads * (DEPTH - 3)));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        issue(s + DEPTH - 1, ring[(u + DEPTH - 1) % DEPTH]);
        read(ring[(u + 1) % DEPTH], xv[(u + 1) & 1], wv[(u + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);  // the reads go out before the MFMAs that hide them
        mfma(xv[u & 1], wv[u & 1]);
    };
    // Whole trips without a branch between stages: where paths join, the
    // compiler waits for the most recent loads of either.
    constexpr int kTrip = DEPTH % 2 == 0 ? DEPTH : 2 * DEPTH;  // ring slots and register sets are constants
    int s = 0;
    for (; s + kTrip <= stages; s += kTrip) {
#pragma unroll
        for (int u = 0; u < kTrip; ++u) {
            stage_step(s + u, u);
        }
    }
#pragma unroll
    for (int u = 0; u < kTrip - 1; ++u) {
        if (s + u < stages) {
            stage_step(s + u, u);
        }
    }
    __builtin_amdgcn_s_waitcnt(kWaitVm(0));  // every load to LDS has landed before the ring is reused
    __syncthreads();
    // Exchange: wave q finishes quarter q of the accumulators.  `ex` holds, for
    // each source wave, quarter and accumulator, four chains of 64 lanes; the
    // stage arrays are carved into 4-KB blocks.
    constexpr int kBlocksPerStage = T::kStageFloats / 1024;
    auto block = [&](int b) -> float* {  // b is a constant once unrolled
        return ring[b / kBlocksPerStage] + b % kBlocksPerStage * 1024;
    };
    static_assert(4 * T::kQuarter <= kBlocksPerStage * DEPTH, "a round of the exchange fits the ring");
    float ls[T::kQuarter][8];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        // block (quarter, i): source wave s at 256 s + 4 lane
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
            for (int i = 0; i < T::kQuarter; ++i) {
                f32x4 v;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    v[j] = acc[4 * half + j].get(q, i);
                }
                *reinterpret_cast<f32x4*>(block(q * T::kQuarter + i) + wave * 256 + 4 * lane) = v;
            }
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (wave == q) {
#pragma unroll
                for (int i = 0; i < T::kQuarter; ++i) {
                    const float* from = block(q * T::kQuarter + i) + 4 * lane;
                    const f32x4 a0 = *reinterpret_cast<const f32x4*>(from);
                    const f32x4 a1 = *reinterpret_cast<const f32x4*>(from + 256);
                    const f32x4 a2 = *reinterpret_cast<const f32x4*>(from + 512);
                    const f32x4 a3 = *reinterpret_cast<const f32x4*>(from + 768);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        // (a[l] + a[8 + l]) + (a[16 + l] + a[24 + l])
                        ls[i][4 * half + j] = (a0[j] + a1[j]) + (a2[j] + a3[j]);
                    }
                }
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < T::kQuarter; ++i) {
        // lanes j and j + 4, (h0 + h2) + (h1 + h3)
        const float h0 = ls[i][0] + ls[i][4];
        const float h1 = ls[i][1] + ls[i][5];
        const float h2 = ls[i][2] + ls[i][6];
        const float h3 = ls[i][3] + ls[i][7];
        const float total = (h0 + h2) + (h1 + h3);
        const int t = M == 32 ? 8 * wave + 4 * lk + i : 4 * lk + wave;
        const int r = M == 32 ? li : M * i + li;
        const int64_t row = row0 + r;
        const bool live = t < ntok && r < nrow;
        if (live && (!BEST || out != nullptr)) {
            float* o = out + static_cast<int64_t>(t0 + t) * rows + row;
            *o = accumulate ? __builtin_fmaf(scale, total, *o) : total;
        }
        if constexpr (BEST) {
            // the tile's best row of each token: the M lanes that share it, then
            // (16-token tiles) one candidate per 16 rows
            HeadBest b = candidate(total, row, live);
#pragma unroll
            for (int o = M / 2; o >= 1; o >>= 1) {
                const HeadBest other{__shfl_xor(b.v, o), __shfl_xor(b.i, o), __shfl_xor(b.have, o)};
                b = better(b, other);
            }
            if (li == 0 && t < ntok) {
                const int64_t per = static_cast<int64_t>(nr) * NR;
                partial[static_cast<int64_t>(t0 + t) * per + static_cast<int64_t>(rt) * NR + (M == 32 ? 0 : i)] = b;
            }
        }
    }
}

// The same dot product for one token (the projections of a decode step): 32
// lanes per row (dot_bf16_lanes32), two rows per wave, so even a 576-row
// projection spreads over 72 workgroups.
// STEPS > 0: in_dim == 32 STEPS, and every step's weight word and activation
// is loaded before the first multiply-add (the whole matrix in flight at once
// when there are few rows); the chain and the lane reduction are
// dot_bf16_lanes32's.
template <int STEPS>
__global__ __launch_bounds__(256) void matvec_one_kernel(const uint16_t* __restrict__ w, const float* __restrict__ x,
                                                         float* out, int64_t rows, int32_t in_dim, float scale,
                                                         int32_t accumulate) {
    const int lane = threadIdx.x & 63;
    const int c = lane & 31;
    const int64_t row = (static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6)) * 2 + (lane >> 5);
    const bool live = row < rows;
    const uint16_t* wr = w + (live ? row : rows - 1) * in_dim;
    float total;
    if constexpr (STEPS > 0) {
        uint32_t word[STEPS];
        float xv[STEPS];
        const uint32_t* w32 = reinterpret_cast<const uint32_t*>(wr) + (c >> 1);
#pragma unroll
        for (int u = 0; u < STEPS; ++u) {
            word[u] = w32[16 * u];
            xv[u] = x[32 * u + c];
        }
        float acc = 0.0f;
#pragma unroll
        for (int u = 0; u < STEPS; ++u) {
            acc = __builtin_fmaf(bits_float((c & 1) != 0 ? (word[u] & 0xffff0000u) : (word[u] << 16)), xv[u], acc);
        }
        const float t1 = acc + __shfl_xor(acc, 8);
        const float t2 = t1 + __shfl_xor(t1, 16);
        const float t3 = t2 + __shfl_xor(t2, 4);
        const float t4 = t3 + __shfl_xor(t3, 2);
        total = t4 + __shfl_xor(t4, 1);
    } else {
        total = dot_bf16_lanes32(wr, [&](int e) { return x[e]; }, in_dim, c);
    }
    if (live && c == 0) {
        out[row] = accumulate ? __builtin_fmaf(scale, total, out[row]) : total;
    }
}

// Sampler::select_next's greedy branch over the blocks' candidates:
// std::max_element keeps the first of equal values and moves only on a strictly
// larger one, so a NaN never becomes the choice, except at index 0, which
// nothing after it can replace (`candidate`).  0 when every logit is NaN.
__global__ __launch_bounds__(1024) void argmax_first_kernel(const HeadBest* __restrict__ partial, int32_t blocks,
                                                            int32_t* out) {
    __shared__ HeadBest wave_best[16];
    const HeadBest* p = partial + static_cast<int64_t>(blockIdx.x) * blocks;
    HeadBest b{0.0f, 0, 0};
    for (int i = threadIdx.x; i < blocks; i += 1024) {
        b = better(b, p[i]);
    }
    b = wave_better(b);
    if ((threadIdx.x & 63) == 0) {
        wave_best[threadIdx.x >> 6] = b;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        HeadBest r = wave_best[0];
        for (int k = 1; k < 16; ++k) {
            r = better(r, wave_best[k]);
        }
        out[blockIdx.x] = r.have ? r.i : 0;
    }
}

// Tile shapes of matvec_exact_kernel.
enum class ExactShape { k32, k16x2, k16x1 };

bool exact_supported(int64_t in_dim) { return in_dim % 64 == 0; }

// The shape with the least expected time: a start-up part plus a part per round
// of the 256 CUs, in tenths of a microsecond at in_dim 2048 (measured at 576 to
// 102400 rows and 5 to 128 tokens: one round 14.7 / 10.3 / 8.0, two 22.7 / 14.6
// / 9.3 us).  Few tiles end sooner as small ones, which spread over more CUs
// (kv_a, 576 rows x 77 tokens: 6.7 us as 16 x 16 tiles, 14.5 as 32 x 32); many
// tiles do fewer LDS reads per multiply-add as large ones (102400 rows x 32
// tokens, whole calls: 165 us as 32 x 32 tiles, 184 as 16 x 32).
ExactShape exact_shape(int64_t rows, int64_t in_dim, int64_t tokens) {
    if (in_dim % 128 != 0) {
        return ExactShape::k32;
    }
    auto rounds = [&](int64_t m, int64_t r) {
        return (((tokens + m - 1) / m) * ((rows + r - 1) / r) + 255) / 256;
    };
    const int64_t c32 = 70 + 76 * rounds(32, 32), c16x2 = 60 + 43 * rounds(16, 32), c16x1 = 50 + 32 * rounds(16, 16);
    if (c32 <= c16x2 && c32 <= c16x1) {
        return ExactShape::k32;
    }
    return c16x2 <= c16x1 ? ExactShape::k16x2 : ExactShape::k16x1;
}

template <int M, int NR, int DEPTH>
hipError_t launch_exact_shape(const uint16_t* w, const float* x, float* out, HeadBest* partial, int64_t rows,
                              int64_t in_dim, int64_t tokens, float scale, int32_t accumulate, hipStream_t s) {
    const int64_t nt = (tokens + M - 1) / M;
    const int64_t nr = (rows + M * NR - 1) / (M * NR);
    const int64_t grid = (nr + 7) / 8 * 8 * nt;
    if (grid > INT32_MAX || tokens > INT32_MAX) {
        return hipErrorInvalidValue;
    }
    if (partial != nullptr) {
        hipLaunchKernelGGL((matvec_exact_kernel<M, NR, DEPTH, true>), dim3(static_cast<unsigned>(grid)), dim3(256), 0,
                           s, w, x, out, partial, rows, static_cast<int32_t>(in_dim), static_cast<int32_t>(tokens),
                           static_cast<int32_t>(nt), static_cast<int32_t>(nr), scale, accumulate);
    } else {
        hipLaunchKernelGGL((matvec_exact_kernel<M, NR, DEPTH, false>), dim3(static_cast<unsigned>(grid)), dim3(256), 0,
                           s, w, x, out, partial, rows, static_cast<int32_t>(in_dim), static_cast<int32_t>(tokens),
                           static_cast<int32_t>(nt), static_cast<int32_t>(nr), scale, accumulate);
    }
    return hipGetLastError();
}

// `blocks`: candidates per token in `partial` (when given).
hipError_t launch_exact(const uint16_t* w, const float* x, float* out, HeadBest* partial, int64_t* blocks,
                        int64_t rows, int64_t in_dim, int64_t tokens, float scale, int32_t accumulate,
                        hipStream_t s) {
    const ExactShape shape = exact_shape(rows, in_dim, tokens);
    if (blocks != nullptr) {
        *blocks = shape == ExactShape::k16x2 ? (rows + 31) / 32 * 2 : shape == ExactShape::k32 ? (rows + 31) / 32
                                                                                            : (rows + 15) / 16;
    }
    switch (shape) {
        case ExactShape::k32:
            return launch_exact_shape<32, 1, 6>(w, x, out, partial, rows, in_dim, tokens, scale, accumulate, s);
        case ExactShape::k16x2:
            return launch_exact_shape<16, 2, 4>(w, x, out, partial, rows, in_dim, tokens, scale, accumulate, s);
        default:
            return launch_exact_shape<16, 1, 4>(w, x, out, partial, rows, in_dim, tokens, scale, accumulate, s);
    }
}

}  // namespace

int64_t head_batch(int64_t in_dim) {
    if (exact_supported(in_dim)) {
        return kHeadBatch;
    }
    return std::max<int64_t>(1, std::min<int64_t>(kHeadTokens, 16384 / in_dim));
}

int64_t head_candidates(int64_t rows, int64_t in_dim) {
    const int64_t few = kHeadTokens * ((rows + kRows - 1) / kRows);
    // at most one per 16 rows and token with 16-token tiles, one per 32 with 32-token tiles
    return exact_supported(in_dim) ? std::max(few, kHeadBatch * 2 * ((rows + 31) / 32)) : few;
}

hipError_t launch_head(const uint16_t* w, const float* x, float* logits, HeadBest* partial, int32_t* token,
                       int64_t rows, int32_t in_dim, int32_t tokens, hipStream_t s) {
    if (rows <= 0 || tokens <= 0) {
        return hipSuccess;
    }
    if (tokens > head_batch(in_dim) || in_dim <= 0 || in_dim % 8 != 0 || rows > INT32_MAX) {
        return hipErrorInvalidValue;
    }
    int64_t blocks = (rows + kRows - 1) / kRows;
    // The few-token kernel keeps the tokens' rows in LDS.  Where two to four do
    // not fit (widths above 4096), the tiles take them in one launch:
    // [102400, 5120], 4 tokens, 217 us (466 as three tokens and one).
    const size_t lds = sizeof(float) * static_cast<size_t>(tokens) * static_cast<size_t>(in_dim);
    if (tokens > kHeadTokens || lds > 64 * 1024) {
        if (!exact_supported(in_dim)) {
            return hipErrorInvalidValue;
        }
        const hipError_t err = launch_exact(w, x, logits, token != nullptr ? partial : nullptr, &blocks, rows, in_dim,
                                            tokens, 1.0f, 0, s);
        if (err != hipSuccess || token == nullptr) {
            return err;
        }
        hipLaunchKernelGGL(argmax_first_kernel, dim3(static_cast<unsigned>(tokens)), dim3(1024), 0, s, partial,
                           static_cast<int32_t>(blocks), token);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(head_logits_kernel<kThreads>, dim3(static_cast<unsigned>(blocks)), dim3(kThreads), lds, s, w,
                       x, logits, partial, rows, in_dim, tokens, 1.0f, 0);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess || token == nullptr) {
        return err;
    }
    hipLaunchKernelGGL(argmax_first_kernel, dim3(static_cast<unsigned>(tokens)), dim3(1024), 0, s, partial,
                       static_cast<int32_t>(blocks), token);
    return hipGetLastError();
}

bool matvec_rows_supported(int64_t rows, int64_t in_dim) {
    return rows > 0 && rows <= INT32_MAX && in_dim > 0 && in_dim % 8 == 0 && in_dim <= 16384;
}

hipError_t launch_matvec_rows(const uint16_t* w, const float* x, float* out, int64_t rows, int64_t in_dim, float scale,
                              int32_t accumulate, hipStream_t s) {
    if (!matvec_rows_supported(rows, in_dim)) {
        return hipErrorInvalidValue;
    }
    hipLaunchKernelGGL(head_logits_kernel<kThreads>, dim3(static_cast<unsigned>((rows + kRows - 1) / kRows)), dim3(kThreads),
                       sizeof(float) * static_cast<size_t>(in_dim), s, w, x, out, nullptr, rows,
                       static_cast<int32_t>(in_dim), 1, scale, accumulate);
    return hipGetLastError();
}

hipError_t launch_matvec_tokens(const uint16_t* w, const float* x, float* out, int64_t rows, int64_t in_dim,
                                int64_t tokens, float scale, int32_t accumulate, hipStream_t s) {
    if (tokens <= 0) {
        return hipSuccess;
    }
    if (!matvec_rows_supported(rows, in_dim)) {
        return hipErrorInvalidValue;
    }
    if (tokens == 1) {
        if (in_dim == 2048) {
            hipLaunchKernelGGL(matvec_one_kernel<64>, dim3(static_cast<unsigned>((rows + 7) / 8)), dim3(256), 0, s, w,
                               x, out, rows, static_cast<int32_t>(in_dim), scale, accumulate);
        } else {
            hipLaunchKernelGGL(matvec_one_kernel<0>, dim3(static_cast<unsigned>((rows + 7) / 8)), dim3(256), 0, s, w, x,
                               out, rows, static_cast<int32_t>(in_dim), scale, accumulate);
        }
        return hipGetLastError();
    }
    // Few tokens on few rows: the tiles spread 2 to 4 tokens over the CUs too
    // (4096 x 2048, 4 tokens: 8.4 us against 24.7 a row at a time); from some
    // 20,000 rows on, streaming the rows past the vector units is as fast
    // (24576 x 2048, 2 tokens: 24.5 us against 25.0).
    if (exact_supported(in_dim) && (tokens > kHeadTokens || rows <= 16384)) {
        return launch_exact(w, x, out, nullptr, nullptr, rows, in_dim, tokens, scale, accumulate, s);
    }
    // tokens per launch: at most kHeadTokens, and their rows must fit 64 KiB of LDS
    const int64_t per = std::min<int64_t>(kHeadTokens, std::max<int64_t>(1, 16384 / in_dim));
    const int64_t rows_per_block = kRowsPerWave * (kSmallThreads / 64);
    const unsigned blocks = static_cast<unsigned>((rows + rows_per_block - 1) / rows_per_block);
    for (int64_t t0 = 0; t0 < tokens; t0 += per) {
        const int32_t n = static_cast<int32_t>(std::min<int64_t>(per, tokens - t0));
        hipLaunchKernelGGL(head_logits_kernel<kSmallThreads>, dim3(blocks), dim3(kSmallThreads),
                           sizeof(float) * static_cast<size_t>(n) * static_cast<size_t>(in_dim), s, w,
                           x + t0 * in_dim, out + t0 * rows, nullptr, rows, static_cast<int32_t>(in_dim), n, scale,
                           accumulate);
        const hipError_t err = hipGetLastError();
        if (err != hipSuccess) {
            return err;
        }
    }
    return hipSuccess;
}

}  // namespace lm
