// mfma_tile.h -- the pipelined fp16 MFMA tile of the GEMM kernels (k_mfma.hip,
// k_proj.hip): operand rows in panel layout staged straight to LDS, STAGES
// deep, and multiplied on v_mfma_f32_32x32x16_f16.  Each file that includes it
// gets its own types (anonymous namespace), and each kernel a type of its own
// (MODE).
#ifndef LITEMIND_MFMA_TILE_H
#define LITEMIND_MFMA_TILE_H

#include "lm_internal.h"

namespace lm {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int BK = kPanel;                   // halves: 64-byte rows, 4 chunks of 16 B
constexpr int kRowBytes = BK * 2;
constexpr int kXcds = 8;

template <int WM, int WN, int MI, int NJ, int STAGES>
struct Shape {
    static constexpr int WAVES = WM * WN;
    static constexpr int kThreads = 64 * WAVES;
    static constexpr int BM = 32 * WM * MI;            // rows of operand A per tile
    static constexpr int BN = 32 * WN * NJ;            // rows of operand B
    static constexpr int kABytes = BM * kRowBytes;
    static constexpr int kBBytes = BN * kRowBytes;
    static constexpr int kStageBytes = kABytes + kBBytes;
    static constexpr int AL = kABytes / 1024 / WAVES;  // A loads (1 KB wave instructions) per wave per stage
    static constexpr int BL = kBBytes / 1024 / WAVES;
    static constexpr int L = AL + BL;
    static constexpr int NR = MI + NJ;                 // fragment reads per half step
    static constexpr int NP = (MI * NJ + 1) / 2;       // MFMA pairs per half step
    static_assert(AL * 1024 * WAVES == kABytes && AL >= 1, "whole A instructions per wave");
    static_assert(BL * 1024 * WAVES == kBBytes && BL >= 1, "whole B instructions per wave");
    static constexpr int RP = NR <= 2 * NP ? 2 : (NR + NP - 1) / NP;  // second half step's reads per MFMA pair
    static_assert(STAGES >= 3 && STAGES <= 6 && (STAGES - 2) * L < 64, "pipeline depth, vmcnt");
    static_assert(STAGES * kStageBytes <= 80 * 1024, "two workgroups per CU");
};

// Chunk permutation of row r (row bits 1..3 only).  A ds_read_b128 serves 16
// lanes per cycle from 64 banks: lanes 0..15 read rows r0..r0+15 (r0 a
// multiple of 16) at one logical chunk, and the rows that share a bank phase
// (r mod 4) get four different chunk positions; the same holds for 8-lane
// groups over 32 banks.
__device__ inline int row_swizzle(int r) { return ((r >> 2) & 3) ^ (r & 2); }
// LDS byte offset of the 16-byte chunk c of row r.
__device__ inline int chunk_offset(int r, int c) { return r * kRowBytes + ((c ^ row_swizzle(r)) << 4); }

// s_waitcnt with only vmcnt (expcnt and lgkmcnt at their maxima)
#define LM_WAIT_VM(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | (((n) >> 4) << 14) | 0x0F70)

// The per-wave state of a tile and the steps of its pipeline.  One type per
// kernel instantiation (MODE is a parameter).
template <int MODE, int WM, int WN, int MI, int NJ, int STAGES>
struct Tile {
    using Z = Shape<WM, WN, MI, NJ, STAGES>;
    __amdgpu_buffer_rsrc_t ra, rb;  // operand A (token rows / activations), operand B (weight rows)
    unsigned va[Z::AL], vb[Z::BL];  // this lane's byte offset of its row chunk in stage 0
    unsigned a_step, b_step;        // bytes between consecutive K panels
    int lane, wave, wm, wn;
    int blocks;                     // this wave's 32-row blocks holding group rows (0..MI); the rest skip their MFMAs
    half8 fa[2][MI], fb[2][NJ];     // fragments of the two half steps of a stage
    floatx16 acc[MI][NJ];

    // Load q of this wave's stage loads (A first, then B): 1 KB, 16 rows of 64
    // bytes, into LDS by a buffer load (the stage offset is a scalar).
    __device__ void load1(int ks, char* buf, int q) {
        if (q < Z::AL) {
            buffer_lds16(ra, buf + (Z::WAVES * q + wave) * 1024, va[q], static_cast<unsigned>(ks) * a_step);
        } else {
            buffer_lds16(rb, buf + Z::kABytes + (Z::WAVES * (q - Z::AL) + wave) * 1024, vb[q - Z::AL],
                        static_cast<unsigned>(ks) * b_step);
        }
    }
    // Fragment r of half step kk: A blocks 0..MI-1, then B blocks 0..NJ-1.
    __device__ void read1(const char* buf, int kk, int r) {
        const int c = 2 * kk + (lane >> 5);
        if (r < MI) {
            fa[kk][r] = *reinterpret_cast<const half8*>(buf + chunk_offset(wm * 32 * MI + 32 * r + (lane & 31), c));
        } else {
            fb[kk][r - MI] = *reinterpret_cast<const half8*>(
                buf + Z::kABytes + chunk_offset(wn * 32 * NJ + 32 * (r - MI) + (lane & 31), c));
        }
    }
    // MFMAs t and t + 1 of half step kk (of one A block when NJ is even), skipped
    // for a block past the group's rows (its accumulators are never stored).
    __device__ void mma2(int t, int kk) {
        const int i = t / NJ, j = t % NJ;
        if constexpr (NJ % 2 == 0) {
            if (i < blocks) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[kk][i], fb[kk][j], acc[i][j], 0, 0, 0);
                acc[i][j + 1] =
                    __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[kk][i], fb[kk][j + 1], acc[i][j + 1], 0, 0, 0);
            }
        } else {
#pragma unroll
            for (int u = t; u < t + 2 && u < MI * NJ; ++u) {
                acc[u / NJ][u % NJ] =
                    __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[kk][u / NJ], fb[kk][u % NJ], acc[u / NJ][u % NJ], 0, 0, 0);
            }
        }
    }
    // s_waitcnt vmcnt(n L): n later stages of this wave's loads may stay in flight.
    __device__ void wait_stages(int n) {
        if (n >= 4) {
            LM_WAIT_VM(4 * Z::L);
        } else if (n == 3) {
            LM_WAIT_VM(3 * Z::L);
        } else if (n == 2) {
            LM_WAIT_VM(2 * Z::L);
        } else if (n == 1) {
            LM_WAIT_VM(Z::L);
        } else {
            LM_WAIT_VM(0);
        }
    }
    // Stage ks: wait for this wave's loads of it (`behind` later stages stay in
    // flight), barrier (every wave's loads visible; the buffer of stage ks - 1,
    // which the loads of stage ks + STAGES - 1 overwrite, read by every wave),
    // the first half step's fragments, then its MFMAs with the second half
    // step's fragment reads and the stage's loads between them, then the second
    // half step's MFMAs with the remaining loads.  With one read or load
    // between two MFMAs the wave's MFMA issue never waits for a run of memory
    // instructions to be accepted (measured on a dense 4096^3 GEMM: 1,150 cycles
    // per stage against 1,561 with the loads and reads issued in runs).
    __device__ void stage(int ks, const char* cur, char* tgt, bool issue, int behind) {
        wait_stages(behind);
        __builtin_amdgcn_s_barrier();
#pragma unroll
        for (int r = 0; r < Z::NR; ++r) {
            read1(cur, 0, r);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int p = 0; p < 2 * Z::NP; ++p) {
            if (p < Z::NP) {
#pragma unroll
                for (int r = Z::RP * p; r < Z::RP * (p + 1); ++r) {
                    if (r < Z::NR) {
                        read1(cur, 1, r);
                    }
                }
            }
#pragma unroll
            for (int q = p * Z::L / (2 * Z::NP); q < (p + 1) * Z::L / (2 * Z::NP); ++q) {
                if (issue) {
                    load1(ks + STAGES - 1, tgt, q);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            mma2(2 * (p % Z::NP), p / Z::NP);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // All nk stages.  Stages 0 .. STAGES - 2 are in flight before the first;
    // stage ks lives in buffer ks % STAGES and the loads of stage ks + STAGES - 1
    // go to buffer (ks - 1) % STAGES.  A K shorter than STAGES - 1 stages reloads
    // the last stage into buffers that are never read, so every path has the
    // same loads in flight.
    __device__ void run(char* const (&bufs)[6], int nk) {
#pragma unroll
        for (int d = 0; d < STAGES - 1; ++d) {
#pragma unroll
            for (int q = 0; q < Z::L; ++q) {
                load1(d < nk ? d : nk - 1, bufs[d], q);
            }
        }
        int ks = 0;
        for (; ks + 2 * STAGES - 1 <= nk; ks += STAGES) {
#pragma unroll
            for (int j = 0; j < STAGES; ++j) {
                stage(ks + j, bufs[j], bufs[(j + STAGES - 1) % STAGES], true, STAGES - 2);
            }
        }
#pragma unroll
        for (int j = 0; j < 2 * STAGES - 1; ++j) {
            const int kj = ks + j;
            if (kj < nk) {
                const int later = nk - 1 - kj;
                stage(kj, bufs[j % STAGES], bufs[(j + STAGES - 1) % STAGES], kj + STAGES - 1 < nk,
                        later < STAGES - 2 ? later : STAGES - 2);
            }
        }
    }
};

}  // namespace
}  // namespace lm

#endif
