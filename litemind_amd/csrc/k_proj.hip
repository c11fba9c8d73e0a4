// k_proj.hip -- the projections of a prompt's attention on MFMA, each with the
// step that follows it as the GEMM's epilogue, for the head widths of the
// one-launch core (k_flash.hip: 128 + 64 key channels, 128 value channels).
//
// Reference: the projections, rotary step and cache append of
// Attention::forward (src/Attention.cpp:33-75), within the MFMA path's
// tolerance: fp16 operands, fp32 sums, everything after a sum in fp32.
//
//   query    q_proj or q_b: rotary step, then fp16 rows for the core
//   kv       kv_b: the new entries into the fp32 cache and the core's fp16 copies
//   plain    q_a, kv_a: fp32 rows;  o_proj: fp32 rows stored or added
//
// Operand A of a tile is weight rows and operand B token rows, so a lane holds
// one token and groups of four successive channels: rotary pairs meet in a
// lane, and the key cache (channel-major) is written 32 tokens at a time.
// Projections of the same input run as segments of one launch.  There is no
// split of K: small tiles keep a prompt of a few hundred tokens on all CUs
// instead (q and kv_a at 256 tokens: 228 tiles of 64 x 64), which saves the
// partial sums' round trip and the launch that adds them.
#include "lm_internal.h"
#include "mfma_tile.h"

#include <algorithm>

namespace lm {
namespace {

constexpr int kNope = 128;
constexpr int kRope = 64;
constexpr int kQk = kNope + kRope;
constexpr int kVh = 128;

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ inline half4 to_half4(f32x4 v) {
    return half4{static_cast<_Float16>(v[0]), static_cast<_Float16>(v[1]), static_cast<_Float16>(v[2]),
                 static_cast<_Float16>(v[3])};
}

// Where key slot j of a 64-key tile lies in the core's value rows (k_flash.hip).
__device__ inline int value_slot(int j) { return (j & 48) + (j & 4) * 2 + (j & 8) / 2 + (j & 3); }

// Four channels n .. n + 3 (n % 4 == 0) of token t.
__device__ inline void store_query(const ProjArgs& a, int64_t t, int n, f32x4 v) {
    const int h = n / kQk, d = n - h * kQk;
    _Float16* const row = a.q16 + (t * a.heads + h) * kQk;
    const int64_t pos = a.pos0 + t;
    if (d < kNope || pos >= a.max_positions) {
        *reinterpret_cast<half4*>(row + d) = to_half4(v);
        return;
    }
    const int i = (d - kNope) / 2;  // two pairs
    const float2 c = *reinterpret_cast<const float2*>(a.cos_t + pos * (kRope / 2) + i);
    const float2 s = *reinterpret_cast<const float2*>(a.sin_t + pos * (kRope / 2) + i);
    float l0, h0, l1, h1;
    rotate_pair(v[0], v[1], c.x, s.x, l0, h0);
    rotate_pair(v[2], v[3], c.y, s.y, l1, h1);
    *reinterpret_cast<half2v*>(row + kNope + i) = half2v{static_cast<_Float16>(l0), static_cast<_Float16>(l1)};
    *reinterpret_cast<half2v*>(row + kNope + kRope / 2 + i) =
        half2v{static_cast<_Float16>(h0), static_cast<_Float16>(h1)};
}

__device__ inline void store_kv(const ProjArgs& a, int64_t t, int n, f32x4 v) {
    const int h = n / (kNope + kVh), j = n - h * (kNope + kVh);
    const int64_t slot = a.slot0 + t;
    if (j < kNope) {
        float* const key = a.cache.key_nope + (static_cast<int64_t>(h) * kNope + j) * a.cap + slot;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            key[e * a.cap] = v[e];
        }
        *reinterpret_cast<half4*>(a.kv.nope16 + (h * a.kv.kp + slot) * kNope + j) = to_half4(v);
        return;
    }
    const int c = j - kNope;
    *reinterpret_cast<f32x4*>(a.cache.value + (h * a.cap + slot) * kVh + c) = v;
    const int in = static_cast<int>(slot & 63);
    _Float16* const tile = a.kv.v16 + (h * a.kv.kp + (slot - in)) * kVh + value_slot(in);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        tile[(c + e) * 64] = static_cast<_Float16>(v[e]);
    }
}

__device__ inline void store_plain(const ProjSegment& seg, int64_t t, int n, f32x4 v) {
    f32x4* const out = reinterpret_cast<f32x4*>(seg.out + t * seg.rows + n);
    *out = seg.accumulate ? *out + v : v;
}

// SHAPE tells the instantiations' tile types apart.
template <int SHAPE, int WM, int WN, int MI, int NJ, int STAGES>
__global__ __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(2, 2))) void proj_kernel(ProjArgs a) {
    using Z = Shape<WM, WN, MI, NJ, STAGES>;
    // One LDS array per stage: the compiler tracks the asynchronous LDS writes
    // per array.
    __shared__ __attribute__((aligned(1024))) char s0[Z::kStageBytes], s1[Z::kStageBytes], s2[Z::kStageBytes],
        s3[STAGES > 3 ? Z::kStageBytes : 16], s4[STAGES > 4 ? Z::kStageBytes : 16],
        s5[STAGES > 5 ? Z::kStageBytes : 16];
    char* const bufs[6] = {s0, s1, s2, s3, s4, s5};
    Tile<SHAPE, WM, WN, MI, NJ, STAGES> t;
    t.lane = threadIdx.x & 63;
    t.wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    t.wm = t.wave / WN;
    t.wn = t.wave % WN;
    const int lane = t.lane, wave = t.wave;
    // XCD b % 8 takes a contiguous eighth of the tiles, the token tiles of one
    // weight tile together: each weight row comes into one L2.
    const int ntt = static_cast<int>((a.tokens + Z::BN - 1) / Z::BN);
    const int nw0 = (a.seg[0].rows + Z::BM - 1) / Z::BM;
    const int nw1 = (a.seg[1].rows + Z::BM - 1) / Z::BM;
    const int total = (nw0 + nw1) * ntt;
    const int xcd = static_cast<int>(blockIdx.x) % kXcds, idx = static_cast<int>(blockIdx.x) / kXcds;
    const int per = total / kXcds, extra = total % kXcds;
    if (idx >= per + (xcd < extra ? 1 : 0)) {
        return;
    }
    const int tile = xcd * per + std::min(xcd, extra) + idx;
    int wt = tile / ntt;
    const int tt = tile - wt * ntt;
    const bool second = wt >= nw0;
    const ProjSegment seg = second ? a.seg[1] : a.seg[0];
    wt -= second ? nw0 : 0;
    const int K = a.width;
    const int chunk = (lane & 3) ^ row_swizzle(lane >> 2);
    t.ra = __builtin_amdgcn_make_buffer_rsrc((void*)seg.w, 0, static_cast<int>(static_cast<int64_t>(seg.rows) * K * 2),
                                             kBufferWord3);
    t.rb = __builtin_amdgcn_make_buffer_rsrc((void*)a.x16, 0, static_cast<int>(a.tokens * K * 2), kBufferWord3);
#pragma unroll
    for (int q = 0; q < Z::AL; ++q) {
        const int n = wt * Z::BM + 16 * (Z::WAVES * q + wave) + (lane >> 2);
        t.va[q] = static_cast<unsigned>((std::min(n, seg.rows - 1) * kPanel + chunk * 8) * 2);
    }
#pragma unroll
    for (int q = 0; q < Z::BL; ++q) {
        const int64_t m = static_cast<int64_t>(tt) * Z::BN + 16 * (Z::WAVES * q + wave) + (lane >> 2);
        t.vb[q] = static_cast<unsigned>((std::min<int64_t>(m, a.tokens - 1) * kPanel + chunk * 8) * 2);
    }
    t.a_step = static_cast<unsigned>(seg.rows) * kRowBytes;
    t.b_step = static_cast<unsigned>(a.tokens) * kRowBytes;
    t.blocks = MI;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            t.acc[i][j] = floatx16{};
        }
    }
    t.run(bufs, K / BK);
    // Lane l holds token l % 32 of each block and channels 8 g + 4 (l / 32) .. + 3
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int64_t token = static_cast<int64_t>(tt) * Z::BN + t.wn * (32 * NJ) + 32 * j + (lane & 31);
        if (token >= a.tokens) {
            continue;
        }
#pragma unroll
        for (int i = 0; i < MI; ++i) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int n = wt * Z::BM + t.wm * (32 * MI) + 32 * i + 8 * g + 4 * (lane >> 5);
                if (n >= seg.rows) {
                    continue;
                }
                const f32x4 v = {t.acc[i][j][4 * g], t.acc[i][j][4 * g + 1], t.acc[i][j][4 * g + 2],
                                 t.acc[i][j][4 * g + 3]};
                if (seg.kind == kProjQuery) {
                    store_query(a, token, n, v);
                } else if (seg.kind == kProjKv) {
                    store_kv(a, token, n, v);
                } else {
                    store_plain(seg, token, n, v);
                }
            }
        }
    }
}

// gemm::rms_norm of rows of `cols` (the first cols of rows `stride` apart) into
// fp16 panels, from the rounded fp32 values as to_f16_rows_kernel converts
// them.  cols % 8 == 0.
__device__ inline void norm16_row(const float* row, const float* w, _Float16* out16, int64_t r, int64_t rows,
                                  int cols, float eps, double* part) {
    const float inverse = rms_inverse_256(row, cols, eps, part);
    for (int c = 8 * static_cast<int>(threadIdx.x); c < cols; c += 8 * 256) {
        half8 out;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            f32x4 v = *reinterpret_cast<const f32x4*>(row + c + 4 * u);
            const f32x4 nw = *reinterpret_cast<const f32x4*>(w + c + 4 * u);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float x = v[e] * inverse;
                x = x * nw[e];
                asm volatile("" : "+v"(x));  // round to fp32 first: no mixed-precision product
                out[4 * u + e] = static_cast<_Float16>(x);
            }
        }
        *reinterpret_cast<half8*>(out16 + panel_index(r, c, rows)) = out;
    }
}

__global__ __launch_bounds__(256) void norm16_kernel(const float* __restrict__ in, const float* __restrict__ w,
                                                     _Float16* __restrict__ out16, int64_t rows, int32_t cols,
                                                     float eps) {
    __shared__ double part[4];
    norm16_row(in + blockIdx.x * static_cast<int64_t>(cols), w, out16, blockIdx.x, rows, cols, eps, part);
}

// Workgroup t < tokens: kv_prep_kernel's step for one token (k_attn.hip) with
// the normalised latent as fp16 panels, and the rotary key into the fp32 cache
// and the core's copy.  Workgroup tokens + h: zeros into head h's values past
// the call's last key, up to the end of their tile (their probabilities are
// zero, and zero times a stale infinity would not be).
__global__ __launch_bounds__(256) void kv_prep16_kernel(const ProjArgs a, const float* __restrict__ lat,
                                                        const float* __restrict__ norm_w,
                                                        _Float16* __restrict__ kvn16, int32_t rank, float eps) {
    __shared__ double part[4];
    const int64_t t = blockIdx.x;
    if (t >= a.tokens) {
        const int h = static_cast<int>(t - a.tokens);
        const int64_t keys = a.slot0 + a.tokens;
        const int from = static_cast<int>(keys & 63);
        if (from == 0) {
            return;
        }
        _Float16* const tile = a.kv.v16 + (h * a.kv.kp + (keys - from)) * kVh;
        for (int i = threadIdx.x; i < 64 * kVh; i += 256) {
            const int in = i & 63;
            if (in >= from) {
                tile[(i >> 6) * 64 + value_slot(in)] = static_cast<_Float16>(0.0f);
            }
        }
        return;
    }
    const float* const row = lat + t * static_cast<int64_t>(rank + kRope);
    norm16_row(row, norm_w, kvn16, t, a.tokens, rank, eps, part);
    const int64_t pos = a.pos0 + t;
    const int64_t slot = a.slot0 + t;
    const int i = threadIdx.x;
    if (i < kRope / 2) {
        const float e = row[rank + 2 * i];
        const float o = row[rank + 2 * i + 1];
        float lo = e, hi = o;
        int at_lo = 2 * i, at_hi = 2 * i + 1;  // positions past the table stay as they are
        if (pos < a.max_positions) {
            rotate_pair(e, o, a.cos_t[pos * (kRope / 2) + i], a.sin_t[pos * (kRope / 2) + i], lo, hi);
            at_lo = i;
            at_hi = i + kRope / 2;
        }
        a.cache.key_rope[at_lo * a.cap + slot] = lo;
        a.cache.key_rope[at_hi * a.cap + slot] = hi;
        a.kv.rope16[slot * kRope + at_lo] = static_cast<_Float16>(lo);
        a.kv.rope16[slot * kRope + at_hi] = static_cast<_Float16>(hi);
    }
}

// Tile shape (weight rows x tokens): 0: 64 x 64, 1: 64 x 128, 2: 128 x 128,
// 3: 128 x 256.  The largest that still gives two thirds of the CUs a tile, and
// 64 x 128 once the 64 x 64 tiles would queue up.  Measured (V2-Lite, us for
// shapes 0 / 1 / 2 / 3): q and kv_a, 256 tokens 10.6 / 14 / 20 / 33, 777 27 / 24
// / 23 / 36, 2048 74 / 54 / 43 / 42, 4096 143 / 144 / 89 / 77; o_proj, 512 tokens
// 8.8 / 11 / 15 / 24, 1024 15 / 13 / 16 / 25, 2048 39 / 24 / 20 / 28.
int proj_shape(int64_t rows, int64_t tokens) {
    auto tiles = [&](int64_t m, int64_t n) { return ((rows + m - 1) / m) * ((tokens + n - 1) / n); };
    if (tiles(128, 256) >= 170) {
        return 3;
    }
    if (tiles(128, 128) >= 170) {
        return 2;
    }
    return tiles(64, 64) > 384 ? 1 : 0;
}

template <int SHAPE, int WM, int WN, int MI, int NJ, int STAGES>
hipError_t launch_proj_shape(const ProjArgs& a, hipStream_t s) {
    using Z = Shape<WM, WN, MI, NJ, STAGES>;
    int64_t tiles = 0;
    for (const ProjSegment& seg : a.seg) {
        tiles += (seg.rows + Z::BM - 1) / Z::BM * ((a.tokens + Z::BN - 1) / Z::BN);
    }
    const int64_t grid = (tiles + kXcds - 1) / kXcds * kXcds;
    if (grid > INT32_MAX) {
        return hipErrorInvalidValue;
    }
    hipLaunchKernelGGL((proj_kernel<SHAPE, WM, WN, MI, NJ, STAGES>), dim3(static_cast<unsigned>(grid)),
                       dim3(Z::kThreads), 0, s, a);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_proj(const ProjArgs& a, hipStream_t s) {
    if (a.tokens <= 0) {
        return hipSuccess;
    }
    const int64_t limit = 0x7fffffff;
    if (a.width <= 0 || a.width % BK != 0 || a.tokens * a.width * 2 > limit) {
        return hipErrorInvalidValue;
    }
    int64_t rows = 0;
    for (const ProjSegment& seg : a.seg) {
        if (seg.rows % 4 != 0 || static_cast<int64_t>(seg.rows) * a.width * 2 > limit) {
            return hipErrorInvalidValue;
        }
        rows += seg.rows;
    }
    switch (proj_shape(rows, a.tokens)) {
        case 0:
            return launch_proj_shape<0, 2, 2, 1, 1, 6>(a, s);
        case 1:
            return launch_proj_shape<1, 2, 2, 1, 2, 5>(a, s);
        case 2:
            return launch_proj_shape<2, 2, 2, 2, 2, 4>(a, s);
        default:
            return launch_proj_shape<3, 2, 2, 2, 4, 3>(a, s);
    }
}

hipError_t launch_norm16(const float* in, const float* w, _Float16* out16, int64_t rows, int32_t cols, float eps,
                         hipStream_t s) {
    if (rows <= 0) {
        return hipSuccess;
    }
    hipLaunchKernelGGL(norm16_kernel, dim3(static_cast<unsigned>(rows)), dim3(256), 0, s, in, w, out16, rows, cols,
                       eps);
    return hipGetLastError();
}

hipError_t launch_kv_prep16(const ProjArgs& a, const float* lat, const float* norm_w, _Float16* kvn16, int32_t rank,
                            float eps, hipStream_t s) {
    if (a.tokens <= 0) {
        return hipSuccess;
    }
    hipLaunchKernelGGL(kv_prep16_kernel, dim3(static_cast<unsigned>(a.tokens + a.heads)), dim3(256), 0, s, a, lat,
                       norm_w, kvn16, rank, eps);
    return hipGetLastError();
}

}  // namespace lm
