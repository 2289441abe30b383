// vedic_gemm_f32s.hpp -- the fp32 GEMM on the bf16 matrix cores (gfx950).
//
//   C[M x N] = epi(op(A) . op(B)), A, B and C binary32, op NN / NT / TN, every
//   operand value split exactly into three bf16 parts (vedic_split.hpp), six
//   v_mfma_f32_32x32x16_bf16 per 32 x 32 x 16 block.
//
// Bound: the matrix cores, 6 x 2 M N K bf16 operations.  An element is split
// once per workgroup that reads it, as it goes from registers to LDS, so the
// split's VALU work (5.5 instructions per element and the scaling) stays a
// third of the MFMA time of a 128 x 128 tile and runs beside it.
//
// A workgroup: one BM x BN tile, WGM x WGN waves.  Per stage (16 contraction
// steps): the fp32 values of stage k + 2 are loaded into registers, those of
// stage k + 1 are split and written to the other of two LDS buffers, and stage
// k's fragments feed 6 MI NI MFMAs; one barrier per stage.  LDS per buffer is
// 96 (BM + BN) bytes, 24 KiB at 128 x 128, so three workgroups share a CU
// (three waves per SIMD): one's staging and epilogue run under the others'
// MFMAs, and no persistent loop is needed.
//
// LDS rows: one per output row / column, 96 bytes: part p at 32 p, 16
// contraction steps of 2 bytes in two 16-byte halves, half h stored at
// h ^ bit 3 of the row.  A 16-lane ds_read_b128 (16 rows, one half) then
// starts at 16-byte groups 6 r mod 16 (+ 1 for rows 8..15): all 16 distinct.
//
// Staging by layout: contraction contiguous (A in NN / NT, B in NT), eight
// steps of one row per thread by two 16-byte loads (VEC), or two steps per
// thread by 4-byte loads where rows are not 16-byte aligned; M / N contiguous
// (the others), eight 4-byte loads down one column, coalesced across the
// lanes, so those operands need no alignment at all.
#pragma once

#include <type_traits>

#include "vedic_gemm_f16.hpp"
#include "vedic_split.hpp"

namespace vedic {

constexpr int kSplitK = 16;         // contraction steps per stage
constexpr int kSplitRowBytes = 96;  // 3 parts x 16 steps x 2 bytes
// Sums of one or two products are repeated on the fp32 MFMA: the terms that the
// split drops cost more there than its longer accumulation gains (largest error
// of K = 1, 2, 3 in units of 2^-24 of the summed magnitudes 2.5, 2.8, 2.4 against
// 1.0, 1.95, 2.5).
constexpr int kSplitMinK = 3;

__device__ __forceinline__ int split_half(int row, int h) { return (h ^ ((row >> 3) & 1)) << 4; }

// One operand's staging: R rows of the tile, NT threads.
template <bool KC, bool VEC, int R, int NT>
struct SideSplit {
    // KC VEC and MC: units of eight steps of one row; KC scalar: pairs of steps
    static constexpr bool PAIRS = KC && !VEC;
    static constexpr int UNITS = PAIRS ? R * 8 : R * 2;
    static constexpr int U = (UNITS + NT - 1) / NT;  // per thread
    static constexpr int PER = PAIRS ? 2 : 8;        // values per unit
    static_assert(UNITS % NT == 0, "units divide among the threads");
    uint32_t off[U];  // byte offset of the unit from the stage base; kOob outside M / N
    int k0[U];        // the unit's first step in the stage (uniform per wave for MC)

    typedef float Values[U][PER];  // one stage's values of this thread

    __device__ __forceinline__ static int row_of(int tid, int i) {
        const int u = i * NT + tid;
        return PAIRS ? u >> 3 : KC ? u >> 1 : u % R;
    }
    __device__ __forceinline__ void init(int tid, int64_t ld, int mn0, int MN) {
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int u = i * NT + tid, row = row_of(tid, i);
            // (MC: R is a multiple of the wave size)
            k0[i] = PAIRS ? 2 * (u & 7) : KC ? 8 * (u & 1) : 8 * __builtin_amdgcn_readfirstlane(u / R);
            const bool ok = mn0 + row < MN;
            off[i] = !ok ? kOob : KC ? (uint32_t)((int64_t)row * ld * 4 + k0[i] * 4) : (uint32_t)(row * 4);
        }
    }
    // One stage's values from its base, element (mn0, k) (KC) or (k, mn0) (MC).
    // FULL: all 16 steps, or (steps = 0) none; otherwise `steps` of them, maybe
    // 0 or less.  Steps the stage does not have load as zeros, without
    // touching memory.
    template <bool FULL>
    __device__ __forceinline__ void load(Values& v, const float* base, int64_t ld, int steps) const {
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<float*>(KC ? base : base + (int64_t)k0[i] * ld), 0, !FULL || steps > 0 ? 0x7FFFFFFF : 0,
                0x00020000);
            if constexpr (KC && VEC) {
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const uint32_t o = FULL || k0[i] + 4 * q < steps ? off[i] : kOob;
                    const float4_t w = __builtin_bit_cast(
                        float4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(o == kOob ? kOob : o + 16 * q), 0, 0));
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[i][4 * q + e] = w[e];
                }
            } else if constexpr (KC) {
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const uint32_t o = FULL || k0[i] + e < steps ? off[i] : kOob;
                    v[i][e] = ld_f32(rs, o == kOob ? kOob : o + 4 * e, 0);
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    v[i][e] = ld_f32(rs, FULL || k0[i] + e < steps ? off[i] : kOob, (uint32_t)e * (uint32_t)ld * 4);
            }
        }
    }
    // Splits the values into the stage buffer `lds` (this operand's rows).
    __device__ __forceinline__ void commit(const Values& v, char* lds, int tid) const {
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int row = row_of(tid, i);
            char* dst = lds + row * kSplitRowBytes + split_half(row, k0[i] >> 3);
            if constexpr (PAIRS) {
                const SplitPair s = split_pair(v[i][0] * kSplitScale, v[i][1] * kSplitScale);
#pragma unroll
                for (int p = 0; p < 3; ++p) *reinterpret_cast<uint32_t*>(dst + 32 * p + (k0[i] & 7) * 2) = s.p[p];
            } else {
                float w[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) w[e] = v[i][e] * kSplitScale;
                const SplitFrag f = split8(w);
#pragma unroll
                for (int p = 0; p < 3; ++p) *reinterpret_cast<bf16x8_t*>(dst + 32 * p) = f.p[p];
            }
        }
    }
};

// The operand parts of rows rc0 + lane % 32, steps 8 (lane / 32) .. + 7.
__device__ __forceinline__ SplitFrag read_split(const char* lds, int rc0, int lane) {
    const int row = rc0 + (lane & 31);
    const char* p = lds + row * kSplitRowBytes + split_half(row, lane >> 5);
    SplitFrag f;
#pragma unroll
    for (int q = 0; q < 3; ++q) f.p[q] = *reinterpret_cast<const bf16x8_t*>(p + 32 * q);
    return f;
}

// A wave's (32 MI) x (32 NI) block on v_mfma_f32_32x32x2_f32 from unscaled
// global values: for blocks whose split sums are not finite (an operand of
// 2^104 or more, an infinity, a NaN, a result past 2^80) and for one or two
// steps.  No LDS, no barrier: 2 Q steps' values of all the block's rows and
// columns are in flight together (lane half h takes steps Q h .. Q h + Q - 1 of
// them; Q = 4 where the accumulators leave no more registers), and feed Q MI NI
// MFMAs.  8192 x 8192 x 1024 all NaN NN / NT / TN 5732 /
// 7513 / 3797 -> 1853 / 1618 / 1996 us, of which the split pass is 605 (1003 / 963 /
// 1066 on gemm_f32_kernel); one NaN 2817 / 2585 / 2339 -> 1063 / 916 / 1152.
template <bool A_KC, bool B_KC, int MI, int NI>
__device__ __forceinline__ void f32_block_slow(const GemmArgs& args, int row0, int col0, int kb, int ke, int lane,
                                               float16_t (&acc)[MI][NI]) {
    constexpr int Q = MI * NI > 4 ? 4 : 8;
    const int l32 = lane & 31, h = lane >> 5;
    const float* A = static_cast<const float*>(args.A);
    const float* B = static_cast<const float*>(args.B);
    const int64_t ka = A_KC ? 1 : args.lda, kn = B_KC ? 1 : args.ldb;
    const float* pa[MI];
    const float* pb[NI];
    // (rows and columns past M and N repeat the last: not stored)
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const int r = min(row0 + 32 * i + l32, args.M - 1);
        pa[i] = (A_KC ? A + (int64_t)r * args.lda : A + r) + (kb + Q * h) * ka;
    }
#pragma unroll
    for (int j = 0; j < NI; ++j) {
        const int n = min(col0 + 32 * j + l32, args.N - 1);
        pb[j] = (B_KC ? B + (int64_t)n * args.ldb : B + n) + (kb + Q * h) * kn;
    }
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = float16_t{};
    int k = kb;
#pragma unroll 1
    for (; k + 2 * Q <= ke; k += 2 * Q) {
        float x[MI][Q], y[NI][Q];
#pragma unroll
        for (int i = 0; i < MI; ++i) {
#pragma unroll
            for (int q = 0; q < Q; ++q) x[i][q] = pa[i][q * ka];
            pa[i] += 2 * Q * ka;
        }
#pragma unroll
        for (int j = 0; j < NI; ++j) {
#pragma unroll
            for (int q = 0; q < Q; ++q) y[j][q] = pb[j][q * kn];
            pb[j] += 2 * Q * kn;
        }
#pragma unroll
        for (int q = 0; q < Q; ++q)
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NI; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[i][q], y[j][q], acc[i][j], 0, 0, 0);
    }
    // the last steps, fewer than 2 Q: those past the end load the last one and count as zeros
#pragma unroll 1
    for (int q = 0; q < Q && k + q < ke; ++q) {
        const bool in = k + Q * h + q < ke;
        const int64_t d = in ? q : ke - 1 - (k + Q * h);
        float x[MI], y[NI];
#pragma unroll
        for (int i = 0; i < MI; ++i) x[i] = pa[i][d * ka];
#pragma unroll
        for (int j = 0; j < NI; ++j) y[j] = pb[j][d * kn];
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NI; ++j)
                acc[i][j] =
                    __builtin_amdgcn_mfma_f32_32x32x2f32(in ? x[i] : 0.0f, in ? y[j] : 0.0f, acc[i][j], 0, 0, 0);
    }
}

template <int OP, bool VEC, int BM, int BN, int WGM, int WGN, int WPE, int SETS, int KIND>
__global__ void __launch_bounds__(WGM* WGN * 64) __attribute__((amdgpu_waves_per_eu(WPE)))
gemm_f32s_kernel(GemmArgs args) {
    constexpr int NT = WGM * WGN * 64, WM = BM / WGM, WN = BN / WGN, MI = WM / 32, NI = WN / 32;
    constexpr bool A_KC = OP != 2, B_KC = OP == 1;
    constexpr int BYTES = (BM + BN) * kSplitRowBytes;
    // VALU instructions placed after each MFMA: the split's 7 per element
    constexpr int VPM = (7 * (BM + BN) * kSplitK / NT + kSplitProducts * MI * NI - 1) / (kSplitProducts * MI * NI);
    // (two objects: reads of one stage provably do not alias the writes of the next)
    __shared__ __attribute__((aligned(1024))) char buf0[BYTES];
    __shared__ __attribute__((aligned(1024))) char buf1[BYTES];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int wm = wave / WGN, wn = wave % WGN;
    const int G = gridDim.x, b = blockIdx.x;
    const int w = (G & 7) == 0 ? (b & 7) * (G >> 3) + (b >> 3) : b;
    const WorkItem it = work_of<BM, BN, kSplitK>(args, w, args.tiles_m * args.tiles_n);
    const float* A = static_cast<const float*>(args.A) + (A_KC ? (int64_t)it.m0 * args.lda + it.kb
                                                               : (int64_t)it.kb * args.lda + it.m0);
    const float* B = static_cast<const float*>(args.B) + (B_KC ? (int64_t)it.n0 * args.ldb + it.kb
                                                               : (int64_t)it.kb * args.ldb + it.n0);
    const int64_t ka = A_KC ? 1 : args.lda, kb = B_KC ? 1 : args.ldb;  // elements per step

    // Stage kt's values wait in register set kt % SETS, its parts in LDS
    // buffer kt % 2.  Stages come in groups of P; the first P take the slice's
    // remainder past whole groups (1 .. 16 P steps, the earlier ones maybe
    // none), so that every later stage is full, its loads carry no bounds
    // arithmetic, and the loop has no tail.
    constexpr int P = SETS < 2 ? 2 : SETS;
    static_assert(P % 2 == 0, "whole pairs of LDS buffers");
    using SA = SideSplit<A_KC, VEC, BM, NT>;
    using SB = SideSplit<B_KC, VEC, BN, NT>;
    SA sa;
    SB sb;
    sa.init(tid, args.lda, it.m0, args.M);
    sb.init(tid, args.ldb, it.n0, args.N);
    // (len 0, no stage at all, for the steps that f32_block_slow does alone)
    const bool few = it.ke - it.kb < kSplitMinK;
    const int len = few ? 0 : it.ke - it.kb, nk = (len + P * kSplitK - 1) / (P * kSplitK) * P;
    const int rem = few ? 0 : len - (nk - P) * kSplitK;
    typename SA::Values va[SETS];
    typename SB::Values vb[SETS];
    auto load_first = [&](int kt) {  // kt < P
        const int b0 = max(0, rem - (P - kt) * kSplitK), b1 = max(0, rem - (P - 1 - kt) * kSplitK);
        sa.template load<false>(va[kt % SETS], A + b0 * ka, args.lda, b1 - b0);
        sb.template load<false>(vb[kt % SETS], B + b0 * kb, args.ldb, b1 - b0);
    };
    auto load = [&](int set, int kt) {  // kt >= P; none past the range
        const int64_t k = rem + (int64_t)(kt - P) * kSplitK;
        const int steps = kt < nk ? kSplitK : 0;
        sa.template load<true>(va[set], A + k * ka, args.lda, steps);
        sb.template load<true>(vb[set], B + k * kb, args.ldb, steps);
    };
    auto commit = [&](int set, char* buf) {
        sa.commit(va[set], buf, tid);
        sb.commit(vb[set], buf + BM * kSplitRowBytes, tid);
    };

    float16_t acc[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = float16_t{};

    auto read = [&](const char* cur, SplitFrag (&fa)[MI], SplitFrag (&fb)[NI]) {
#pragma unroll
        for (int j = 0; j < NI; ++j) fb[j] = read_split(cur + BM * kSplitRowBytes, wn * WN + 32 * j, lane);
#pragma unroll
        for (int i = 0; i < MI; ++i) fa[i] = read_split(cur, wm * WM + 32 * i, lane);
    };
    auto multiply = [&](const SplitFrag (&fa)[MI], const SplitFrag (&fb)[NI]) {
#pragma unroll
        for (int q = 0; q < kSplitProducts; ++q)
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NI; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i].p[kSplitA[q]], fb[j].p[kSplitB[q]],
                                                                        acc[i][j], 0, 0, 0);
    };
    // Multiplies the stage in `cur`, splits the next one's values into `nxt`
    // (free since the last barrier) and loads those of stage kt into their
    // place.
    auto stage = [&](const char* cur, char* nxt, int set, int kt) {
        SplitFrag fa[MI], fb[NI];
        read(cur, fa, fb);
        commit(set, nxt);
        load(set, kt);
        multiply(fa, fb);
        // the fragment reads, then a few VALU instructions of the split (and
        // an LDS write once there is one) after every MFMA
        __builtin_amdgcn_sched_group_barrier(0x100, 3 * (MI + NI), 0);
#pragma unroll
        for (int x = 0; x < kSplitProducts * MI * NI; ++x) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, VPM, 0);
            __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        stage_barrier();
    };
#pragma unroll
    for (int q = 0; q < SETS; ++q) {
        load_first(q);
        __builtin_amdgcn_sched_barrier(0);  // loads in flight in the loop's order
    }
    commit(0, buf0);
    if constexpr (SETS < P) load_first(SETS);
    else load(0, SETS);
    stage_barrier();
    for (int kt = 0; kt < nk; kt += P) {
#pragma unroll
        for (int q = 0; q < P; ++q)
            stage(q & 1 ? buf1 : buf0, q & 1 ? buf0 : buf1, (q + 1) % SETS, kt + q + 1 + SETS);
    }

    const int row0 = it.m0 + wm * WM, col0 = it.n0 + wn * WN;
    float probe = 0.0f;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            acc[i][j] *= kSplitUnscale2;
            probe = nonfinite_probe(acc[i][j], probe);
        }
    if (few || __any(probe != 0.0f))
        f32_block_slow<A_KC, B_KC, MI, NI>(args, row0, col0, it.kb, it.ke, lane, acc);
    // split-K: this slice's raw partial goes to its own slab of the workspace
    void* const cp = args.ksplit > 1 ? static_cast<void*>(static_cast<float*>(args.C) + it.s * args.c_split_stride)
                                   : args.C;
    const bool full = (row0 + WM <= args.M) && (col0 + WN <= args.N);
    if (KIND != EK_GENERIC && full)
        epilogue<KIND, false, MI, NI, kStoreDevice>(args, cp, acc, row0, col0, lane);
    else
        epilogue<KIND, true, MI, NI, kStoreDevice>(args, cp, acc, row0, col0, lane);
}

// Tile configurations.  Waves per SIMD (WPE) follow the registers: 128
// accumulators per lane of the 256 x 256 tile leave two.  8192 x 8192 x 1024 NN
// 595 us with 256 x 256 tiles (231 TFLOP/s; 1005 us on v_mfma_f32_32x32x2_f32),
// 647 with 128 x 128: half the LDS reads and splits per MFMA, the matrix pipe
// busy 69 % of the active cycles.  One
// workgroup of 128 x 128 per CU reaches 177 TFLOP/s (4096 x 1024 x 8192).
struct CfgSLarge {  // 256 x 256, eight waves of 128 x 64, one workgroup per CU
    static constexpr int BM = 256, BN = 256, WGM = 2, WGN = 4, WPE = 2, SETS = 1;
};
struct CfgSMid {  // 128 x 128, four waves of 64 x 64, three workgroups per CU
    static constexpr int BM = 128, BN = 128, WGM = 2, WGN = 2, WPE = 3, SETS = 1;
};
// 64 x 64, two waves of 32 x 64, for few output tiles with unaligned rows (the
// aligned ones run on v_mfma_f32_32x32x2_f32): four stages of loads in
// flight, since with one or two workgroups per CU a stage is only as long as
// its own 12 MFMAs.
struct CfgSSmall {
    static constexpr int BM = 64, BN = 64, WGM = 2, WGN = 1, WPE = 2, SETS = 4;
};

template <int OP, bool VEC, class Cfg, int KIND>
static hipError_t launch_f32s(GemmArgs a, hipStream_t s) {
    a.tiles_m = (a.M + Cfg::BM - 1) / Cfg::BM;
    a.tiles_n = (a.N + Cfg::BN - 1) / Cfg::BN;
    if (a.group_m <= 0) a.group_m = 8;
    if (a.ksplit < 1) {
        a.ksplit = 1;
        a.kslice = a.K;
    }
    const int nwork = a.tiles_m * a.tiles_n * a.ksplit;
    hipLaunchKernelGGL((gemm_f32s_kernel<OP, VEC, Cfg::BM, Cfg::BN, Cfg::WGM, Cfg::WGN, Cfg::WPE, Cfg::SETS, KIND>), dim3(nwork),
                       dim3(Cfg::WGM * Cfg::WGN * 64), 0, s, a);
    return hipGetLastError();
}

// Rows that are not 16-byte aligned (VEC false) run the generic epilogue; TN
// loads its operands element-wise whatever their alignment.
template <int OP, bool VEC, class Cfg>
static hipError_t launch_f32s_kind(const GemmArgs& a, hipStream_t s) {
    if constexpr (VEC) {
        switch (a.epi_kind) {
            case EK_PLAIN: return launch_f32s<OP, VEC, Cfg, EK_PLAIN>(a, s);
            case EK_BIAS: return launch_f32s<OP, VEC, Cfg, EK_BIAS>(a, s);
            case EK_BIAS_GELU: return launch_f32s<OP, VEC, Cfg, EK_BIAS_GELU>(a, s);
            case EK_BIAS_GELU_PRE: return launch_f32s<OP, VEC, Cfg, EK_BIAS_GELU_PRE>(a, s);
            case EK_ACCUM: return launch_f32s<OP, VEC, Cfg, EK_ACCUM>(a, s);
            case EK_GELU_BWD: return launch_f32s<OP, VEC, Cfg, EK_GELU_BWD>(a, s);
            case EK_LINEAR_CS: return launch_f32s<OP, VEC, Cfg, EK_LINEAR_CS>(a, s);
            case EK_RESIDUAL: return launch_f32s<OP, VEC, Cfg, EK_RESIDUAL>(a, s);
        }
    }
    return launch_f32s<OP, VEC, Cfg, EK_GENERIC>(a, s);
}

#define VEDIC_F32S_KERNEL(OP, VEC, Cfg, KIND) \
    template __global__ void gemm_f32s_kernel<OP, VEC, Cfg::BM, Cfg::BN, Cfg::WGM, Cfg::WGN, Cfg::WPE, Cfg::SETS, KIND>(GemmArgs)
#define VEDIC_F32S_KINDS(OP, Cfg)                         \
    VEDIC_F32S_KERNEL(OP, true, Cfg, EK_PLAIN);           \
    VEDIC_F32S_KERNEL(OP, true, Cfg, EK_BIAS);            \
    VEDIC_F32S_KERNEL(OP, true, Cfg, EK_BIAS_GELU);       \
    VEDIC_F32S_KERNEL(OP, true, Cfg, EK_BIAS_GELU_PRE);   \
    VEDIC_F32S_KERNEL(OP, true, Cfg, EK_ACCUM);           \
    VEDIC_F32S_KERNEL(OP, true, Cfg, EK_GELU_BWD);        \
    VEDIC_F32S_KERNEL(OP, true, Cfg, EK_LINEAR_CS);       \
    VEDIC_F32S_KERNEL(OP, true, Cfg, EK_RESIDUAL);        \
    VEDIC_F32S_KERNEL(OP, true, Cfg, EK_GENERIC)

// 256 x 256 tiles where their whole rounds cost less than the 128 x 128 tiles'
// share per CU: a 256 x 256 round does four 128 x 128 tiles' work at 1.1 times
// their rate (8192 x 8192 above; 8192 x 3072, 1.5 rounds, 254 against 246 us).
// Not for contractions of at most 64, which the writing of C bounds: three
// workgroups on a CU overlap their epilogues, one does not (8192 x 4096 NT
// accumulated, K = 4 59.0 us against 42.0, 64 65.9 / 47.4; 8192 x 8192 K = 4 59.9 /
// 44.1, 64 75.4 / 72.0, 128 108.5 / 108.3, 256 176.4 / 186.3).
inline bool f32s_large(int M, int N, int K, int cus) {
    if (K <= 64) return false;
    const int64_t t256 = (int64_t)((M + 255) / 256) * ((N + 255) / 256);
    const int64_t t128 = (int64_t)((M + 127) / 128) * ((N + 127) / 128);
    return (t256 + cus - 1) / cus * 4 * 10 < (t128 + cus - 1) / cus * 11;
}

template <int OP, bool VEC>
hipError_t launch_gemm_f32s_op(const GemmArgs& a, hipStream_t s) {
    const int cus = device_cu_count();
    if constexpr (VEC) {
        // (256 rows of a longer leading dimension pass 32-bit offsets)
        if (a.ksplit <= 1 && a.lda < kMaxLd / 2 && a.ldb < kMaxLd / 2 && f32s_large(a.M, a.N, a.K, cus))
            return launch_f32s_kind<OP, VEC, CfgSLarge>(a, s);
        if constexpr (OP != 2) return launch_f32s_kind<OP, VEC, CfgSMid>(a, s);
    }
    // (TN, whose kernels take any alignment, and unaligned rows: few tiles too)
    if (!f32s_mid_tiles(a.M, a.N, a.K, cus)) return launch_f32s_kind<OP, VEC, CfgSSmall>(a, s);
    return launch_f32s_kind<OP, VEC, CfgSMid>(a, s);
}

}  // namespace vedic
