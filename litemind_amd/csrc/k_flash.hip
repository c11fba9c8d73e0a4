// k_flash.hip -- the attention core of a batch of query tokens in one launch
// (fp16 operands, fp32 sums), for heads of 128 + 64 key channels and 128 value
// channels (DeepSeek-V2 and V2-Lite).
//
// Reference: the scores, softmax and context of Attention::forward
// (src/Attention.cpp:77-98), within the MFMA path's tolerance: queries, keys
// and values rounded to fp16, every sum in fp32, the probabilities
// exp(scale (s - m)) rounded to fp16 as the second product's operand and
// summed unrounded.
//
// The scores never leave the registers.  A wave owns 32 query tokens of one
// head and walks the cached keys in tiles of 64: S^T = K Q^T, so that each
// lane holds the scores of one query (column lane % 32; the two half waves
// hold alternate groups of four keys), the running maximum and total are one
// value per lane, and the probabilities of a lane are already the B operand of
// ctx^T = V^T P^T, whose K order is free: the values are stored with the keys
// of each group of 16 in the order in which the lanes hold them.  Waves of a
// workgroup share the key and value tiles, staged straight to LDS two tiles
// deep, 16-byte units XOR-swizzled by row so that the fragment reads are free
// of bank conflicts.
//
// Few query tokens over many keys would leave most CUs idle: the keys are then
// split over several workgroups, whose unnormalised contexts, maxima and
// totals flash_combine_kernel joins.
#include "lm_internal.h"

#include <algorithm>

namespace lm {
namespace {

constexpr int kNope = 128;
constexpr int kRope = 64;
constexpr int kQk = kNope + kRope;
constexpr int kVh = 128;
constexpr int NW = 4;                           // waves of 32 query tokens per workgroup
constexpr int kBlock = 32 * NW;                 // query tokens per workgroup
constexpr int kTile = 64;                       // keys per tile
constexpr int kNopeBytes = kTile * kNope * 2;   // 16 KB
constexpr int kRopeBytes = kTile * kRope * 2;   // 8 KB
constexpr int kValueBytes = kTile * kVh * 2;    // 16 KB

typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// ---- fp16 copies of the cache ----
//   nope16    [heads][Kp][128]           row j = key_nope(h, :, j)
//   rope16    [Kp][64]                   row j = key_rope(:, j), shared by the heads
//   values16  [heads][Kp / 64][128][64]  value(h, j, :) transposed per tile of 64
//                                        keys, each 16 in the order 0-3, 8-11,
//                                        4-7, 12-15: half wave h's scores are
//                                        keys 4 h .. + 3 and 8 + 4 h .. + 3, its k
//                                        indices 8 h .. + 7 of the second product
// Kp = the call's keys rounded up to 64.  New entries are written as they are
// computed (k_proj.hip); flash_pack_kernel copies the `keys` older ones, zeros
// up to the end of their last tile.  Workgroup (tile, head), the head past the
// last for rope16.
__global__ __launch_bounds__(256) void flash_pack_kernel(const float* __restrict__ key_nope,
                                                         const float* __restrict__ key_rope,
                                                         const float* __restrict__ value, const FlashKv kv,
                                                         int32_t heads, int64_t cap, int64_t keys) {
    __shared__ float tile[kTile * (kVh + 1)];  // keys: [64 channels][65]; values: [64 keys][129]
    const int tid = threadIdx.x;
    const int64_t j0 = static_cast<int64_t>(blockIdx.x) * kTile;
    const int h = blockIdx.y;
    const bool rope = h == heads;
    const int width = rope ? kRope : kNope;
    const float* const src = rope ? key_rope : key_nope + static_cast<int64_t>(h) * kNope * cap;
    _Float16* const rows = rope ? kv.rope16 + j0 * kRope : kv.nope16 + (static_cast<int64_t>(h) * kv.kp + j0) * kNope;
    for (int p = 0; p < width / 64; ++p) {  // 64 channels at a time
        float v[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int64_t j = std::min<int64_t>(j0 + (tid & 63), keys - 1);
            v[i] = src[(p * 64 + i * 4 + (tid >> 6)) * cap + j];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            tile[(i * 4 + (tid >> 6)) * 65 + (tid & 63)] = v[i];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int kk = (tid >> 3) + 32 * i, part = tid & 7;
            half8 out;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                out[e] = j0 + kk < keys ? static_cast<_Float16>(tile[(part * 8 + e) * 65 + kk])
                                        : static_cast<_Float16>(0.0f);
            }
            *reinterpret_cast<half8*>(rows + kk * width + p * 64 + part * 8) = out;
        }
    }
    if (rope) {
        return;
    }
    f32x4 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int64_t j = std::min<int64_t>(j0 + i * 8 + (tid >> 5), keys - 1);
        v[i] = *reinterpret_cast<const f32x4*>(value + (static_cast<int64_t>(h) * cap + j) * kVh + (tid & 31) * 4);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            tile[(i * 8 + (tid >> 5)) * (kVh + 1) + (tid & 31) * 4 + e] = v[i][e];
        }
    }
    __syncthreads();
    _Float16* const dst = kv.v16 + (static_cast<int64_t>(h) * kv.kp + j0) * kVh;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c = (tid >> 3) + 32 * i, part = tid & 7;  // positions 8 part .. + 7 of channel c
        half8 out;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int pos = (part & 1) * 8 + e;  // within the group of 16
            const int k = part / 2 * 16 + (pos & 3) + (pos & 4) * 2 + (pos & 8) / 2;
            out[e] = j0 + k < keys ? static_cast<_Float16>(tile[k * (kVh + 1) + c]) : static_cast<_Float16>(0.0f);
        }
        *reinterpret_cast<half8*>(dst + c * kTile + part * 8) = out;
    }
}

struct FlashArgs {
    const _Float16* q16;   // [T][heads][192], rotary applied
    FlashKv kv;
    _Float16* ctx16;       // panels [ctx_rows][heads 128] (one split)
    float* part_o;         // [splits][heads][T][128] unnormalised contexts (several splits)
    float* part_ml;        // [splits][heads][T][2] maximum and total
    int64_t T, n0;
    int64_t row0, ctx_rows;
    int32_t heads, qblocks, splits, split_tiles;
    float c;               // softmax scale times log2(e)
};

template <bool SPLIT>
__global__ __launch_bounds__(64 * NW, 2) void flash_kernel(const FlashArgs a) {
    __shared__ __align__(16) char k0[kNopeBytes], k1[kNopeBytes], r0[kRopeBytes], r1[kRopeBytes], v0[kValueBytes],
        v1[kValueBytes];
    char* const kring[2] = {k0, k1};
    char* const rring[2] = {r0, r1};
    char* const vring[2] = {v0, v1};
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    // Workgroup -> (head, query block, split).  Heads are dealt to the XCDs
    // (workgroup ids go round robin over them), so a head's tiles come into
    // one L2; the blocks with the most keys go first, and a launch that fits
    // the chip at two workgroups per CU pairs them with the lightest.
    const int xcd = static_cast<int>(blockIdx.x) & 7;
    int local = static_cast<int>(blockIdx.x) >> 3;
    const int hpx = (a.heads + 7) / 8;
    const int h = xcd + 8 * (local % hpx);
    local /= hpx;
    const int split = SPLIT ? local % a.splits : 0;
    const int order = SPLIT ? local / a.splits : local;
    if (h >= a.heads) {
        return;
    }
    const int heavy = (a.qblocks + 1) / 2;
    const int qb = order < heavy ? a.qblocks - 1 - order : order - heavy;
    const int64_t q0 = static_cast<int64_t>(qb) * kBlock;
    const int half = lane >> 5;
    const int64_t qw = q0 + 32 * wave;                              // the wave's first query
    const int64_t qi = qw + (lane & 31);                            // this lane's query
    const int64_t qc = std::min<int64_t>(qi, a.T - 1);
    const int64_t vis = a.n0 + qc;                                  // last key it sees
    const int64_t block_keys = a.n0 + std::min<int64_t>(a.T, q0 + kBlock);
    const int all_tiles = static_cast<int>((block_keys + kTile - 1) / kTile);
    const int tile0 = SPLIT ? split * a.split_tiles : 0;
    const int tile_end = SPLIT ? std::min(all_tiles, tile0 + a.split_tiles) : all_tiles;
    if (SPLIT && tile0 >= tile_end) {
        return;  // the block's keys end before this split (flash_combine_kernel does not read it)
    }
    // tiles this wave has a visible key in; none for waves past the last query
    const int wave_end = qw < a.T ? static_cast<int>((a.n0 + std::min<int64_t>(a.T, qw + 32) + kTile - 1) / kTile) : 0;
    // queries: B operand of S^T, k-step ks holds channels 16 ks + 8 half .. + 7
    half8 qf[kQk / 16];
    {
        const _Float16* qr = a.q16 + (qc * a.heads + h) * kQk + 8 * half;
#pragma unroll
        for (int ks = 0; ks < kQk / 16; ++ks) {
            qf[ks] = *reinterpret_cast<const half8*>(qr + 16 * ks);
        }
    }
    // Tile loads: a load fills 64 consecutive 16-byte positions.  A 16-byte LDS
    // read serves 16 lanes, so 16 successive rows go to 16 different columns of
    // banks: position p of row r holds unit p ^ (r % 16) of the nope keys (256
    // bytes a row, four rows a load) and p ^ (r / 2 % 8) of the rotary keys and
    // the values (128 bytes, eight rows).
    const int64_t head_keys = static_cast<int64_t>(h) * a.kv.kp;
    const __amdgpu_buffer_rsrc_t kres = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.kv.nope16 + head_keys * kNope), 0, static_cast<int>(a.kv.kp * kNope * 2), kBufferWord3);
    const __amdgpu_buffer_rsrc_t rres = __builtin_amdgcn_make_buffer_rsrc(
        (void*)a.kv.rope16, 0, static_cast<int>(a.kv.kp * kRope * 2), kBufferWord3);
    const __amdgpu_buffer_rsrc_t vres = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.kv.v16 + head_keys * kVh), 0, static_cast<int>(a.kv.kp * kVh * 2), kBufferWord3);
    // Load j of a run: the units of load 0 with bits 2 and 3 (4 j % 16) flipped.
    const unsigned ksrc = static_cast<unsigned>((lane >> 4) * (kNope * 2) + ((lane & 15) ^ (lane >> 4)) * 16);
    const unsigned vsrc = static_cast<unsigned>((lane >> 3) * 128 + ((lane & 7) ^ (lane >> 4)) * 16);
    auto issue = [&](int tile, char* ks, char* rs, char* vs) {
#pragma unroll
        for (int j = 0; j < 16 / NW; ++j) {
            const int at = wave * (16 / NW) + j;  // a multiple of four, plus j
            buffer_lds16(kres, ks + at * 1024, ksrc ^ (j & 3) * 64u, tile * kNopeBytes + at * 1024);
        }
#pragma unroll
        for (int j = 0; j < 8 / NW; ++j) {
            const int at = wave * (8 / NW) + j;
            buffer_lds16(rres, rs + at * 1024, vsrc ^ (j & 1) * 64u, tile * kRopeBytes + at * 1024);
        }
#pragma unroll
        for (int j = 0; j < 16 / NW; ++j) {
            const int at = wave * (16 / NW) + j;
            buffer_lds16(vres, vs + at * 1024, vsrc ^ (j & 1) * 64u, tile * kValueBytes + at * 1024);
        }
    };
    f32x16 o[kVh / 32] = {};
    float m = -__builtin_inff();  // running maximum of the raw scores
    f32x4 l = {};                 // this half wave's share of the total, in four sums
    auto compute = [&](int tile, const char* ks, const char* rs, const char* vs) {
        f32x16 s[2] = {};
        const int r = lane & 31;
        // Fragments in sets of four (keys: two k-steps of both 32-key halves;
        // values: one k-step of all channels), each read before the MFMAs of
        // the set before it.
        half8 fa[4], fb[4];
        auto read_keys = [&](int g, half8 (&f)[4]) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = 32 * (i & 1) + r, u = 4 * g + 2 * (i >> 1) + half;
                f[i] = *reinterpret_cast<const half8*>(
                    g < kNope / 32 ? ks + row * (kNope * 2) + (u ^ (r & 15)) * 16
                                   : rs + row * (kRope * 2) + ((u - kNope / 8) ^ ((r >> 1) & 7)) * 16);
            }
        };
        auto read_values = [&](int st, half8 (&f)[4]) {
#pragma unroll
            for (int vt = 0; vt < 4; ++vt) {
                f[vt] = *reinterpret_cast<const half8*>(vs + (32 * vt + r) * (kTile * 2) +
                                                        ((2 * st + half) ^ ((r >> 1) & 7)) * 16);
            }
        };
        auto score = [&](int g, const half8 (&f)[4]) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[i], qf[2 * g + (i >> 1)], s[i & 1], 0, 0, 0);
            }
        };
        read_keys(0, fa);
#pragma unroll
        for (int g = 0; g < kQk / 32; g += 2) {
            read_keys(g + 1, fb);
            __builtin_amdgcn_sched_barrier(0);
            score(g, fa);
            __builtin_amdgcn_sched_barrier(0);
            if (g + 2 < kQk / 32) {
                read_keys(g + 2, fa);
            } else {
                read_values(0, fa);
            }
            __builtin_amdgcn_sched_barrier(0);
            score(g + 1, fb);
            __builtin_amdgcn_sched_barrier(0);
        }
        // register e of s[kt] is key 64 tile + 32 kt + 8 (e / 4) + 4 half + e % 4
        if (static_cast<int64_t>(tile + 1) * kTile > a.n0 + qw + 1) {
            const int last = static_cast<int>(vis - static_cast<int64_t>(tile) * kTile);
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    if (32 * kt + 8 * (e / 4) + 4 * half + e % 4 > last) {
                        s[kt][e] = -__builtin_inff();
                    }
                }
            }
        }
        float t4[4];  // four chains
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            t4[e] = fmaxf(s[0][e], s[1][e]);
#pragma unroll
            for (int k = 4; k < 16; k += 4) {
                t4[e] = fmaxf(fmaxf(t4[e], s[0][e + k]), s[1][e + k]);
            }
        }
        float t = fmaxf(fmaxf(t4[0], t4[1]), fmaxf(t4[2], t4[3]));
        t = fmaxf(t, __shfl_xor(t, 32));
        const float m_new = fmaxf(m, t);
        if (__any(m_new > m)) {
            // no key seen yet: any finite reference, every exponential is 0
            const float alpha = m_new == -__builtin_inff() ? 1.0f : __builtin_amdgcn_exp2f((m - m_new) * a.c);
            l *= alpha;
#pragma unroll
            for (int vt = 0; vt < kVh / 32; ++vt) {
                o[vt] *= alpha;
            }
            m = m_new;
        }
        const float mc = m == -__builtin_inff() ? 0.0f : m * a.c;
        // ctx^T += V^T P^T: k-step st covers the 16 keys of registers 8 st .. + 7
        half8 pf;
        auto weights = [&](int st) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[st / 2][8 * (st & 1) + e], a.c, -mc));
                l[e % 4] += p;
                pf[e] = static_cast<_Float16>(p);
            }
        };
        auto context = [&](const half8 (&f)[4]) {
#pragma unroll
            for (int vt = 0; vt < 4; ++vt) {
                o[vt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[vt], pf, o[vt], 0, 0, 0);
            }
        };
#pragma unroll
        for (int st = 0; st < 4; st += 2) {
            read_values(st + 1, fb);
            weights(st);
            context(fa);
            if (st + 2 < 4) {
                read_values(st + 2, fa);
            }
            weights(st + 1);
            context(fb);
        }
    };
    issue(tile0, k0, r0, v0);
    for (int tb = tile0; tb < tile_end; tb += 2) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int tile = tb + u;
            if (tile < tile_end) {
                // the tile is in, and every wave is done with the one before it
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_s_waitcnt(0x0070 | 0x0F00);  // vmcnt(0)
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
                if (tile + 1 < tile_end) {
                    issue(tile + 1, kring[1 - u], rring[1 - u], vring[1 - u]);
                }
                if (tile < wave_end) {
                    compute(tile, kring[u], rring[u], vring[u]);
                }
            }
        }
    }
    float total = (l[0] + l[1]) + (l[2] + l[3]);
    total += __shfl_xor(total, 32);
    if (qi >= a.T) {
        return;
    }
    // o[vt] register e: channel 32 vt + 8 (e / 4) + 4 half + e % 4 of query lane % 32
    if constexpr (SPLIT) {
        const int64_t at = (static_cast<int64_t>(split) * a.heads + h) * a.T + qi;
        if (half == 0) {
            a.part_ml[2 * at] = m;
            a.part_ml[2 * at + 1] = total;
        }
#pragma unroll
        for (int vt = 0; vt < kVh / 32; ++vt) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                f32x4 out;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    out[e] = o[vt][4 * g + e];
                }
                *reinterpret_cast<f32x4*>(a.part_o + at * kVh + 32 * vt + 8 * g + 4 * half) = out;
            }
        }
    } else {
        const float inv = 1.0f / total;
#pragma unroll
        for (int vt = 0; vt < kVh / 32; ++vt) {
            _Float16* row = a.ctx16 + panel_index(a.row0 + qi, h * kVh + 32 * vt, a.ctx_rows) + 4 * half;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                half4 out;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    out[e] = static_cast<_Float16>(o[vt][4 * g + e] * inv);
                }
                *reinterpret_cast<half4*>(row + 8 * g) = out;
            }
        }
    }
}

// The splits' contexts of one (token, head) joined: weights exp(scale (m_i -
// max)), over the weighted total.  32 lanes per (token, head), four channels
// each.
__global__ __launch_bounds__(256) void flash_combine_kernel(const FlashArgs a) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 8 + (threadIdx.x >> 5);
    const int lane = threadIdx.x & 31;
    if (i >= a.T * a.heads) {
        return;
    }
    const int64_t t = i / a.heads;
    const int h = static_cast<int>(i - t * a.heads);
    const int64_t step = a.heads * a.T;
    const int64_t at = h * a.T + t;
    // splits that the token's block of queries has keys in
    const int64_t keys = a.n0 + std::min<int64_t>(a.T, (t / kBlock + 1) * kBlock);
    const int splits = static_cast<int>(((keys + kTile - 1) / kTile + a.split_tiles - 1) / a.split_tiles);
    float m = -__builtin_inff();
    for (int k = 0; k < splits; ++k) {
        m = fmaxf(m, a.part_ml[2 * (at + k * step)]);
    }
    f32x4 o = {};
    float l = 0.0f;
    for (int k = 0; k < splits; ++k) {
        const float w = __builtin_amdgcn_exp2f((a.part_ml[2 * (at + k * step)] - m) * a.c);
        l = __builtin_fmaf(w, a.part_ml[2 * (at + k * step) + 1], l);
        const f32x4 p = *reinterpret_cast<const f32x4*>(a.part_o + (at + k * step) * kVh + 4 * lane);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            o[e] = __builtin_fmaf(w, p[e], o[e]);
        }
    }
    const float inv = 1.0f / l;
    half4 out;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        out[e] = static_cast<_Float16>(o[e] * inv);
    }
    *reinterpret_cast<half4*>(a.ctx16 + panel_index(a.row0 + t, h * kVh + 4 * lane, a.ctx_rows)) = out;
}

}  // namespace

bool flash_supported(const AttnShape& a) { return a.nope == kNope && a.rope == kRope && a.vh == kVh; }

int64_t flash_keys(int64_t keys) { return round_up(keys, kTile); }

// Splits while the query blocks leave CUs idle, of at least four tiles on
// average (a causal block sees half of the call's own keys).  Measured (V2-Lite,
// 16 heads, whole calls in a row on one stream; us for 1 / 2 / 4 / 8 splits): 16
// tokens after 4000 126 / 91 / 73 / 66, 256 after 3000 118 / 89 / 74 / 70, 512
// after 3000 130 / 101 / 86 / 90, 512 alone 54 / 54 / 54 / 58, 1024 alone 80 / 78
// / 80 / 85, after 1000 110 / 100 / 101 / 109, after 20000 595 / 413 / 400 / 412,
// 2048 alone 144 / 146 / 148 / 154.  Workgroups of one or two waves were slower
// throughout: a tile is staged for fewer query tokens.
FlashPlan flash_plan(int32_t heads, int64_t tokens, int64_t keys) {
    FlashPlan p;
    const int64_t tiles = (keys + kTile - 1) / kTile;
    const int64_t blocks = heads * ((tokens + kBlock - 1) / kBlock);
    const int64_t mean = (keys - tokens / 2) / kTile;
    const int64_t want = std::min<int64_t>({16, 256 / blocks, mean / 4});
    p.split_tiles = want > 1 ? static_cast<int32_t>((tiles + want - 1) / want) : 0;
    p.splits = p.split_tiles > 0 ? static_cast<int32_t>((tiles + p.split_tiles - 1) / p.split_tiles) : 1;
    return p;
}

int64_t flash_partial_floats(const FlashPlan& p, int32_t heads, int64_t tokens) {
    return p.splits > 1 ? p.splits * heads * tokens * (kVh + 2) : 0;
}

hipError_t launch_flash_pack(const AttnShape& a, const KvCacheDev& c, int64_t keys, const FlashKv& kv, hipStream_t s) {
    if (keys <= 0) {
        return hipSuccess;
    }
    hipLaunchKernelGGL(flash_pack_kernel, dim3(static_cast<unsigned>((keys + kTile - 1) / kTile), a.heads + 1),
                       dim3(256), 0, s, c.key_nope, c.key_rope, c.value, kv, a.heads, a.cap, keys);
    return hipGetLastError();
}

hipError_t launch_flash(const AttnShape& a, const FlashPlan& p, const _Float16* q16, const FlashKv& kv, float* partial,
                        int64_t T, int64_t n0, float scale, _Float16* ctx16, int64_t row0, int64_t ctx_rows,
                        hipStream_t s) {
    if (T <= 0) {
        return hipSuccess;
    }
    if (!flash_supported(a) || n0 + T > kv.kp || row0 + T > ctx_rows) {
        return hipErrorInvalidValue;
    }
    FlashArgs f;
    f.q16 = q16;
    f.kv = kv;
    f.ctx16 = ctx16;
    f.part_o = partial;
    f.part_ml = partial != nullptr ? partial + p.splits * a.heads * T * kVh : nullptr;
    f.T = T;
    f.n0 = n0;
    f.row0 = row0;
    f.ctx_rows = ctx_rows;
    f.heads = a.heads;
    f.qblocks = static_cast<int32_t>((T + kBlock - 1) / kBlock);
    f.splits = p.splits;
    f.split_tiles = p.split_tiles;
    f.c = scale * 1.4426950408889634f;
    const int64_t grid = (f.heads + 7) / 8 * 8 * static_cast<int64_t>(f.qblocks) * f.splits;
    if (grid > INT32_MAX) {
        return hipErrorInvalidValue;
    }
    if (f.splits == 1) {
        hipLaunchKernelGGL(flash_kernel<false>, dim3(static_cast<unsigned>(grid)), dim3(64 * NW), 0, s, f);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(flash_kernel<true>, dim3(static_cast<unsigned>(grid)), dim3(64 * NW), 0, s, f);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) {
        return err;
    }
    hipLaunchKernelGGL(flash_combine_kernel, dim3(static_cast<unsigned>((T * a.heads + 7) / 8)), dim3(256), 0, s, f);
    return hipGetLastError();
}

}  // namespace lm
