// vedic_flash_attn.hip -- fused attention forward for gfx950, fp32 in and out
// (on the bf16 matrix cores by exact splits, fa_item_split).
//
//   out = softmax(scale * Q . K^T + mask) . V          per head, Q/K/V/out [seq x DH]
//
// the computation of cuda_flash_attention_fwd / flash_attention_kernel
// (cuda/VedicGEMM.cu:898-1104 of the reference): scores masked by causality
// (key > query) and by the optional sparse pattern (keep a key if it lies in
// [query - window, query] or is a multiple of `stride`), masked scores set to
// -1e30 and left out of the sums, an online (running-max) softmax, and a
// final division by the row sum (0 if the sum is <= 1e-9).
//
// Work item: one head, a group of 128 queries (four waves of 32) and a chunk
// of keys.  The workgroup streams the chunk's keys through LDS in blocks of
// 32 (K block and V block together); every wave reuses each block for its own
// 32 queries.  Per block and wave, on the fp32 MFMA (fa_item, the repeat of
// items that the split does not cover; two stages in flight by direct global ->
// LDS loads):
//   S^T [32 keys x 32 queries] = K_blk . Q^T     DH/2 x v_mfma_f32_32x32x2_f32
//   running max / sum update, P = exp(S - max)   (lane l owns query l % 32)
//   O^T [DH x 32 queries]     += V_blk^T . P^T   DH/2 x v_mfma_f32_32x32x2_f32
// Computing the transposed products lets the score accumulator be the PV
// product's B operand without any data movement: the contraction over keys
// is taken in the accumulator's own key order (lane half h, register
// t = 4 g + r holds key 8 g + 4 h + r), and the V reads follow that order.
// The Q . K^T contraction likewise runs over d in the order lane half h,
// step t -> d = (DH/2) h + t, so each lane's Q fragment and K reads are
// contiguous.
//
// When a query group's keys are split over several chunks (single-head calls,
// to spread the work over the CUs) each chunk writes its unnormalised partial
// O with its row max and sum to a workspace, and flash_merge_kernel combines
// the chunks in ascending order.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "vedic_flash_device.hpp"
#include "vedic_flash_split.hpp"

namespace vedic {

template <int DH>
constexpr int fa_stage_bytes() {
    return 2 * kFaKeys * DH * 4;  // one stage: a K block, then a V block
}

#ifndef VEDIC_FA_WPE64
#define VEDIC_FA_WPE64 3
#endif
#ifndef VEDIC_FA_WPE128
#define VEDIC_FA_WPE128 2
#endif
// LDS buffers of the blocks' bf16 parts
template <int DH>
constexpr int fa_buffers() {
    return DH == 64 ? 2 : 1;
}
// LDS stages in flight of the fp32 repeat
template <int DH>
constexpr int fa_stages() {
    return 2;
}

struct FaItem {
    int head, g, k_lo, nkb, nch;
    int64_t asc;
};

// Work item `item` in decreasing size order.
template <int DH>
__device__ __forceinline__ FaItem fa_work(const FlashArgs& a, int item) {
    // Heads interleaved, query groups from the last (largest) down.
    const int head = item % a.nheads;
    const int64_t asc = (int64_t)a.items - 1 - item / a.nheads;
    int lo = 0, hi = a.nqg - 1;  // largest g with prefix(g) <= asc
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (fa_prefix(a, mid) <= asc) lo = mid;
        else hi = mid - 1;
    }
    const int g = lo;
    const int c = (int)(asc - fa_prefix(a, g));
    const int nch = fa_nchunks(a, g);
    const int kend = fa_kend(a, g);
    const int k_lo = c * a.chunk, k_hi = min(kend, k_lo + a.chunk);
    const int nkb = (k_hi - k_lo + kFaKeys - 1) / kFaKeys;
    return {head, g, k_lo, nkb, nch, asc};
}

// An item's results: O / L and the log-sum-exp of its rows, or its slot of
// partials.  l_run holds each lane half's sums; O is `unscale` (a power of two)
// times the accumulators.
template <int DH>
__device__ __forceinline__ void fa_store(const FlashArgs& a, const FaItem& w, const float16_t (&o)[DH / 32], float m_run,
                                         float l_run, float unscale, int wave, int lane) {
    const int l32 = lane & 31, h = lane >> 5;
    const int query = w.g * kFaQ + 32 * wave + l32;
    // Row sums: each lane half summed its own 16 keys per block.
    const float l_tot = l_run + __shfl_xor(l_run, 32);
    // o[d][4 gg + r] is O[query][32 d + 8 gg + 4 h + r].
    if (w.nch == 1) {
        if (query >= a.seq) return;
        if (a.lse[w.head] != nullptr && h == 0) a.lse[w.head][query] = fa_lse(m_run, l_tot);
        const float inv = l_tot > 1e-9f ? 1.0f / l_tot * unscale : 0.0f;
        float* orow = a.o[w.head] + (int64_t)query * DH;
#pragma unroll
        for (int d = 0; d < DH / 32; ++d)
#pragma unroll
            for (int gg = 0; gg < 4; ++gg) {
                float4_t v;
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = o[d][4 * gg + r] * inv;
                store16_hold(orow + 32 * d + 8 * gg + 4 * h, v);
            }
    } else {
        // partial slot: [kFaQ][DH] unnormalised O, then the row maxima and sums
        float* slot = a.part + ((int64_t)w.head * a.items + w.asc) * (kFaQ * DH + 2 * kFaQ);
        float* orow = slot + (int64_t)(32 * wave + l32) * DH;
#pragma unroll
        for (int d = 0; d < DH / 32; ++d)
#pragma unroll
            for (int gg = 0; gg < 4; ++gg) {
                float4_t v;
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = o[d][4 * gg + r] * unscale;
                store16_hold(orow + 32 * d + 8 * gg + 4 * h, v);
            }
        if (h == 0) {
            slot[kFaQ * DH + 32 * wave + l32] = m_run;
            slot[kFaQ * DH + kFaQ + 32 * wave + l32] = l_tot;
        }
    }
}

// One work item (`item` in decreasing size order) with the workgroup's two
// LDS stages t0, t1.
template <int DH>
__device__ __forceinline__ void fa_item(const FlashArgs& a, int item, int tid, char* t0, char* t1) {
    constexpr int KB = kFaKeys * DH * 4;  // bytes of one K (or V) block
    constexpr int SB = fa_stage_bytes<DH>();
    constexpr int NLD = SB / 1024 / 4;    // 1 KiB direct loads per wave per stage
    constexpr int CPR = DH / 4;           // 16-byte chunks per row
    constexpr int HALF = DH / 2;
    static_assert(DH == 64 || DH == 128, "head dimension 64 or 128");
    constexpr int FST = fa_stages<DH>();
    char* const stg[2] = {t0, t1};

    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, l32 = lane & 31, h = lane >> 5;

    const FaItem w = fa_work<DH>(a, item);
    const int head = w.head, g = w.g, k_lo = w.k_lo, nkb = w.nkb;

    const float* __restrict__ Qh = a.q[head];
    const float* __restrict__ Kh = a.k[head];
    const float* __restrict__ Vh = a.v[head];
    const int q0 = g * kFaQ + 32 * wave;  // this wave's first query
    const int query = q0 + l32;           // the query this lane's columns belong to

    // Direct-load geometry (fa_issue): byte offset in the block, row, and K/V part.
    uint32_t loff[NLD];
    int lrow[NLD];
    bool lisv[NLD];
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
        const int ins = wave * NLD + i;
        const bool isv = ins >= KB / 1024;
        const int qq = (isv ? ins - KB / 1024 : ins) * 64 + lane;
        const int row = qq / CPR, pc = qq % CPR;
        // K: chunk c of row m at c ^ (m & 15); V: the two 128-byte halves of a
        // row swapped when bit 2 of the key is set.
        const int cl = isv ? pc ^ (((row >> 2) & 1) * 8) : pc ^ (row & 15);
        loff[i] = (uint32_t)(row * DH * 4 + cl * 16);
        lrow[i] = row;
        lisv[i] = isv;
    }

    // Q fragment: qf[t] = Q[query][HALF * h + t] (zeros past seq).
    float qf[HALF];
    {
        const __amdgpu_buffer_rsrc_t rq = buffer_rsrc(Qh);
        const uint32_t qoff = query < a.seq ? (uint32_t)(query * DH * 4 + HALF * h * 4) : kOob;
#pragma unroll
        for (int j = 0; j < HALF / 4; ++j) {
            // Cast the whole vector to float4: extracting 32-bit integer lanes and
            // casting each to float made this compiler load only lane 0.
            const float4_t v =
                __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(rq, (int)(qoff + 16 * j), 0, 0));
#pragma unroll
            for (int e = 0; e < 4; ++e) qf[4 * j + e] = v[e];
        }
    }

    float16_t o[DH / 32];
#pragma unroll
    for (int d = 0; d < DH / 32; ++d) o[d] = float16_t{};
    // Scores are kept in base 2: s log2(e), so every exponential is one v_exp_f32.
    const float sc2 = a.scale * 1.4426950408889634f;
    float m_run = kFaMasked, l_run = 0.0f;
    const bool wave_live = q0 < a.seq;  // waves past seq only help load

    auto compute = [&](const char* st, int kb) {
        const int key0 = k_lo + kb * kFaKeys;
        if (!wave_live || (a.causal && key0 > q0 + 31)) return;  // every key of the block is masked for this wave
        const char* kl = st;
        const char* vl = st + KB;
        // S^T = K_blk . Q^T: lane (h, l32) supplies K[l32][HALF h + t] and Q[query][HALF h + t].
        float16_t s = float16_t{};
#pragma unroll
        for (int j = 0; j < HALF / 4; ++j) {
            const int cl = (HALF / 4) * h + j;
            const float4_t kf = *reinterpret_cast<const float4_t*>(kl + l32 * DH * 4 + ((cl ^ (l32 & 15)) << 4));
#pragma unroll
            for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[e], qf[4 * j + e], s, 0, 0, 0);
        }
        // s[4 gg + r] is the score of key key0 + 8 gg + 4 h + r for this lane's query.
        const bool need_mask = a.sparse || key0 + kFaKeys > a.seq || (a.causal && key0 + kFaKeys - 1 > q0);
        float mx = kFaMasked;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            float v = s[i] * sc2;
            if (need_mask) v = fa_allowed_score(a, v, key0 + 8 * (i >> 2) + 4 * h + (i & 3), query);
            s[i] = v;
            mx = fmaxf(mx, v);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float m_new = fmaxf(m_run, mx);
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
        float ls = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float p = s[i] <= -1e29f ? 0.0f : __builtin_amdgcn_exp2f(s[i] - m_new);
            s[i] = p;
            ls += p;
        }
        l_run = l_run * alpha + ls;
        m_run = m_new;
#pragma unroll
        for (int d = 0; d < DH / 32; ++d) o[d] *= alpha;
        // O^T += V_blk^T . P^T over the keys in accumulator order: step t pairs
        // key 8 (t/4) + (t%4) (lane half 0) with key 8 (t/4) + 4 + (t%4) (half 1).
#pragma unroll
        for (int d = 0; d < DH / 32; ++d) {
#pragma unroll
            for (int t = 0; t < 16; ++t) {
                const int key = 8 * (t >> 2) + 4 * h + (t & 3);
                const int col = 32 * d + l32;
                const int pcol = (((col >> 2) ^ (h * 8)) << 2) | (col & 3);  // V half swap for keys with bit 2 set
                const float vf = *reinterpret_cast<const float*>(vl + key * DH * 4 + pcol * 4);
                o[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf, s[t], o[d], 0, 0, 0);
            }
        }
    };

#pragma unroll
    for (int st = 0; st < FST - 1; ++st)
        fa_issue<DH, NLD>(Kh, Vh, k_lo + st * kFaKeys, st < nkb ? a.seq - k_lo - st * kFaKeys : 0, stg[st], wave, loff, lrow, lisv);
    for (int k0 = 0; k0 < nkb; k0 += FST) {
#pragma unroll
        for (int st = 0; st < FST; ++st) {
            const int kb = k0 + st;
            wait_vmcnt<(FST - 2) * NLD>();
            stage_barrier();
            {
                const int kn = kb + FST - 1;  // past the range: zeros, no memory touched
                fa_issue<DH, NLD>(Kh, Vh, k_lo + kn * kFaKeys, kn < nkb ? a.seq - k_lo - kn * kFaKeys : 0,
                              stg[(st + FST - 1) % FST], wave, loff, lrow, lisv);
            }
            if (kb < nkb) compute(stg[st], kb);
        }
    }
    wait_vmcnt<0>();  // the trailing zero loads still write LDS
    if (!wave_live) return;
    fa_store<DH>(a, w, o, m_run, l_run, 1.0f, wave, lane);
}

// The same work item on the bf16 matrix cores (vedic_split.hpp): K and V
// blocks are split into three bf16 parts as they go from registers to LDS, Q
// once per item, P in registers.  Per block and wave DH / 16 x 6 MFMAs for S^T and
// DH / 32 x 2 x 6 for O^T, 32 cycles each, against DH of 64 cycles on
// v_mfma_f32_32x32x2_f32: 16 heads x seq 8192 causal 1218 -> 757 us, the
// matrix pipe busy 59 % of the active cycles, 6.4 VALU instructions (split, softmax) per
// MFMA beside it.  scale log2(e) goes into Q before the split, so the
// scores come out in base 2.
//
// Factors against flushed parts (vedic_split.hpp).  Scores: 2^48 on Q, none on
// K (no instruction per key); a part of K below 2^-126 that is lost then meets
// |scale log2(e) Q| < 2^80, an error of a score below 2^-46.  The exponent
// takes the 2^48 out in its subtraction (an fma).  Outputs, which have no scale
// of their own: 2^24 on both P and V (16 heads x seq 8192 +1.6 %).
//
// DH 64: two LDS buffers, one barrier per 32 keys, the block after next in
// flight.  DH 128: a block's parts are 48 KB, so two buffers would leave one
// workgroup per CU, whose splits and softmax nothing overlaps; with one buffer
// and two barriers two workgroups share a CU and one's matrix work covers the
// other's split.  8 heads x seq 8192 causal: fp32 MFMA 1331 us, two buffers
// 943, one 808; 8 x 1000: 51.9, 52.6, 42.2; one head x 8192: 203, 159, 126
// (error against float64 6.3e-7 -> 5.3e-7).
//
// Returns whether the workgroup's results stand.  They do not if a sum is not
// finite or a score is -inf: an infinity or NaN among the operands, a value past
// the split's range (scale log2(e) Q of 2^80, V of 2^104), a score (base 2), a
// partial sum of one, or an output past 2^80.  Then nothing has been written and
// the caller repeats the item with fa_item.
template <int DH>
__device__ __forceinline__ bool fa_item_split(const FlashArgs& a, int item, int tid, char* b0, char* b1) {
    constexpr int KB = fs_block_bytes<DH>();
    constexpr int NT = 256;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, l32 = lane & 31, h = lane >> 5;
    const FaItem w = fa_work<DH>(a, item);
    const float* __restrict__ Kh = a.k[w.head];
    const float* __restrict__ Vh = a.v[w.head];
    const int q0 = w.g * kFaQ + 32 * wave;
    const int query = q0 + l32;
    const bool wave_live = q0 < a.seq;

    SplitFrag qf[DH / 16];
    fs_load_rows<DH>(qf, a.q[w.head], query, a.seq, a.scale * (1.4426950408889634f * kSplitScale * kSplitScale), lane);

    float16_t o[DH / 32];
#pragma unroll
    for (int d = 0; d < DH / 32; ++d) o[d] = float16_t{};
    float m_run = kFaMasked, l_run = 0.0f;
    float low = 0.0f;  // the lowest score, or 0 (-inf would leave l and O finite)

    FsAddr<DH> ad(lane);
    FsStage<DH, NT> sk, sv;
    auto load = [&](int kb) {  // past the range: zeros, no memory touched
        const int key0 = w.k_lo + kb * kFaKeys, rows = kb < w.nkb ? a.seq - key0 : 0;
        sk.load(Kh, key0, rows, tid);
        sv.load(Vh, key0, rows, tid);
    };
    auto commit = [&](char* buf) {
        sk.commit(buf, 1.0f, tid);
        sv.commit(buf + KB, kSplitScale, tid);
    };
    // Keys key0 .. key0 + 31 in `buf`.
    auto compute = [&](const char* buf, int key0) {
        float16_t s = float16_t{};
#pragma unroll
        for (int j = 0; j < DH / 16; ++j) s = mfma_split(fs_row<DH>(buf, ad, j), qf[j], s);
        // s[4 gg + r] is 2^48 times the score of key key0 + 8 gg + 4 h + r for this lane's query.
#pragma unroll
        for (int i = 0; i < 16; ++i) low = fminf(low, s[i]);
        if (a.sparse || key0 + kFaKeys > a.seq || (a.causal && key0 + kFaKeys - 1 > q0)) {
#pragma unroll
            for (int i = 0; i < 16; ++i)
                s[i] = fa_allowed(a, key0 + 8 * (i >> 2) + 4 * h + (i & 3), query) ? s[i] : -__builtin_inff();
        }
        float mx = s[0];
#pragma unroll
        for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
        mx = fmaxf(mx, __shfl_xor(mx, 32)) * kSplitUnscale2;
        if (__any(mx > m_run)) {  // (a factor of 1 for every row otherwise)
            const float m_new = fmaxf(m_run, mx);
            const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
            m_run = m_new;
            l_run *= alpha;
#pragma unroll
            for (int d = 0; d < DH / 32; ++d) o[d] *= alpha;
        }
        // (a masked score's exponential is 0, also in a row with no key yet)
        const float m_ref = m_run == kFaMasked ? 0.0f : m_run;
        float ls = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            s[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], kSplitUnscale2, -m_ref));
            ls += s[i];
        }
        l_run += ls;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const SplitFrag pf = fs_acc(s, j, kSplitScale);
#pragma unroll
            for (int d = 0; d < DH / 32; ++d) o[d] = mfma_split(fs_col<DH>(buf + KB, ad, d, j), pf, o[d]);
        }
    };
    // Whether the wave's queries have a key in block kb (past the item's keys
    // only for an odd count's last step of two buffers).
    auto allowed = [&](int kb) {
        const int key0 = w.k_lo + kb * kFaKeys;
        return wave_live && kb < w.nkb && !(a.causal && key0 > q0 + 31) && !(a.sparse && !fa_sparse_any(a, key0, q0));
    };
    // Step kb: block kb is in `cur`, block kb + 1 in registers.
    auto step = [&](const char* cur, char* nxt, int kb) {
        commit(nxt);
        load(kb + 2);
        ad.refresh();
        if (allowed(kb)) compute(cur, w.k_lo + kb * kFaKeys);
        stage_barrier();
    };

    load(0);
    if constexpr (fa_buffers<DH>() == 1) {
        for (int kb = 0; kb < w.nkb; ++kb) {
            commit(b0);
            load(kb + 1);
            ad.refresh();
            stage_barrier();
            if (allowed(kb)) compute(b0, w.k_lo + kb * kFaKeys);
            stage_barrier();  // every wave is done with the block before the next one overwrites it
        }
    } else {
        commit(b0);
        load(1);
        stage_barrier();
        for (int kb = 0; kb < w.nkb; kb += 2) {
            step(b0, b1, kb);
            step(b1, b0, kb + 1);
        }
    }

    float probe = l_run * 0.0f;
#pragma unroll
    for (int d = 0; d < DH / 32; ++d) probe = nonfinite_probe(o[d], probe);
    if (__syncthreads_or(probe != 0.0f || low == -__builtin_inff())) return false;
    if (wave_live) fa_store<DH>(a, w, o, m_run, l_run, kSplitUnscale2, wave, lane);
    return true;
}

// One work item per workgroup, or (a.queue set) a grid of resident workgroups
// that take items from a counter until none is left: items run largest first,
// so the tail of the key-split one-head case stays balanced.
// DH 64: registers held to three waves per SIMD, the occupancy its 48 KB of
// LDS allows (three workgroups per CU); DH 128: two (two workgroups of 64 KB,
// which the repeat's fp32 stages need).
template <int DH>
__device__ __forceinline__ void fa_run(const FlashArgs& a, int item, char* b0, char* b1) {
    // (The thread index is made opaque for each of the two, so that nothing they
    // derive from it is computed before the loop over items and held in registers
    // across it: 15 and 35 VGPRs spilled at DH 64 and 128 otherwise.)
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    if (fa_item_split<DH>(a, item, tid & 255, b0, b1)) return;
    asm volatile("" : "+v"(tid));
    fa_item<DH>(a, item, tid & 255, b0, b1);
}
template <int DH, bool QUEUE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(DH == 64 ? VEDIC_FA_WPE64 : VEDIC_FA_WPE128)))
flash_attn_kernel(FlashArgs a) {
    // Two LDS objects: reads of one buffer provably do not alias writes of the
    // other.  With one buffer its object holds the repeat's two fp32 stages.
    constexpr bool two = fa_buffers<DH>() == 2;
    constexpr int SB = two ? 2 * fs_block_bytes<DH>() : 2 * fa_stage_bytes<DH>();
    static_assert(SB >= 2 * fs_block_bytes<DH>() && (!two || SB >= fa_stage_bytes<DH>()), "K and V parts; fp32 stages");
    __shared__ __attribute__((aligned(1024))) char b0[SB];
    __shared__ __attribute__((aligned(1024))) char bx[two ? SB : 16];
    char* const b1 = two ? bx : b0 + fa_stage_bytes<DH>();
    __shared__ int next;
    if constexpr (!QUEUE) {
        fa_run<DH>(a, blockIdx.x, b0, b1);
        return;
    }
    const int total = a.items * a.nheads;
    while (true) {
        if (threadIdx.x == 0) next = atomicAdd(a.queue, 1);
        __syncthreads();
        const int item = next;
        __syncthreads();  // every wave has its item before `next` is written again
        if (item >= total) break;
        fa_run<DH>(a, item, b0, b1);
        __syncthreads();  // every wave is done with the stage buffers
    }
}

__global__ void flash_queue_reset(int* queue) {
    if (threadIdx.x == 0) *queue = 0;
}

hipError_t launch_flash_queue_reset(int* queue, hipStream_t s) {
    hipLaunchKernelGGL(flash_queue_reset, dim3(1), dim3(64), 0, s, queue);
    return hipGetLastError();
}

// Combines the chunk partials of every split query group, chunks in
// ascending order with a running maximum M: per chunk c, M' = max(M, m_c),
// L = L 2^(M - M') + l_c 2^(m_c - M'), O likewise; then O / L (row maxima in
// base 2, as the attention kernel keeps them).  The order is fixed, so the
// result does not depend on timing.
// It also returns the work-queue counter to zero for the next queued launch
// on the stream (the attention kernel before it in stream order is done).
template <int DH>
__global__ void __launch_bounds__(256) flash_merge_kernel(FlashArgs a) {
    // one thread per 4 output values; grid (kFaQ DH / 1024, query groups, heads)
    const int g = blockIdx.y, head = blockIdx.z;
    if (a.queue != nullptr && blockIdx.x == 0 && g == 0 && head == 0 && threadIdx.x == 0) *a.queue = 0;
    const int nch = fa_nchunks(a, g);
    if (nch == 1) return;
    const int idx = blockIdx.x * 256 + threadIdx.x;  // < kFaQ * DH / 4
    const int qi = idx / (DH / 4), d4 = idx % (DH / 4);
    const int query = g * kFaQ + qi;
    if (query >= a.seq) return;
    constexpr int SLOT = kFaQ * DH + 2 * kFaQ;
    const float* base = a.part + ((int64_t)head * a.items + fa_prefix(a, g)) * SLOT;
    float M = kFaMasked, L = 0.0f;
    float4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
    // one pass with a running maximum: the chunks' loads are independent and
    // unrolled so they are in flight together; the rescaling is a short chain
#pragma unroll 8
    for (int c = 0; c < nch; ++c) {
        const float* sl = base + (int64_t)c * SLOT;
        const float mc = sl[kFaQ * DH + qi], lc = sl[kFaQ * DH + kFaQ + qi];
        const float4_t oc = *reinterpret_cast<const float4_t*>(sl + qi * DH + 4 * d4);
        const float Mn = fmaxf(M, mc);
        const float so = __builtin_amdgcn_exp2f(M - Mn), w = __builtin_amdgcn_exp2f(mc - Mn);
        L = L * so + lc * w;
        acc = acc * so + oc * w;
        M = Mn;
    }
    const float inv = L > 1e-9f ? 1.0f / L : 0.0f;
    store16_hold(a.o[head] + (int64_t)query * DH + 4 * d4, acc * inv);
    if (a.lse[head] != nullptr && d4 == 0) a.lse[head][query] = fa_lse(M, L);
}

int64_t flash_items_per_head(int seq, int chunk, int causal) {
    FlashArgs a{};
    a.seq = seq;
    a.chunk = chunk;
    a.causal = causal;
    a.nqg = (seq + kFaQ - 1) / kFaQ;
    return fa_prefix(a, a.nqg);
}

int flash_slot_floats(int dh) { return kFaQ * dh + 2 * kFaQ; }

hipError_t launch_flash_attn(const FlashArgs& a, int dh, hipStream_t s) {
    dim3 grid((unsigned)(a.items * a.nheads));
    // (a.queue is zero here: set so when its block was made, and put back by
    // the merge kernel that ends every queued launch)
    if (a.queue != nullptr) grid = dim3((unsigned)std::min(a.items * a.nheads, a.queue_grid));
    const bool q = a.queue != nullptr;
    if (dh == 64) {
        if (q) hipLaunchKernelGGL((flash_attn_kernel<64, true>), grid, dim3(256), 0, s, a);
        else hipLaunchKernelGGL((flash_attn_kernel<64, false>), grid, dim3(256), 0, s, a);
    } else {
        if (q) hipLaunchKernelGGL((flash_attn_kernel<128, true>), grid, dim3(256), 0, s, a);
        else hipLaunchKernelGGL((flash_attn_kernel<128, false>), grid, dim3(256), 0, s, a);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || a.part == nullptr) return e;
    const dim3 mgrid((unsigned)(kFaQ * dh / 4 / 256), (unsigned)a.nqg, (unsigned)a.nheads);
    if (dh == 64) hipLaunchKernelGGL(flash_merge_kernel<64>, mgrid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL(flash_merge_kernel<128>, mgrid, dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace vedic
