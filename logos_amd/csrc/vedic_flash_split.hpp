// vedic_flash_split.hpp -- attention blocks as bf16 parts in LDS, for the
// attention kernels that run on the bf16 matrix cores (vedic_split.hpp).
//
// A block is 32 rows (keys or queries) of DH values, each value as three bf16
// parts.  Row r, part p, 16-byte chunk c (8 values) lies at
//     r * (6 DH) + p * (2 DH) + 16 * (c ^ swz(r)),
// read either along rows (ds_read_b128: an MFMA operand whose contraction is
// over DH) or down columns (two ds_read_b64_tr_b16: one whose contraction is
// over the block's rows).
//   DH 64: rows are 384 bytes, so rows r and r + 1 start in opposite halves of
//   the 256-byte bank window.  Row reads (16 rows, one chunk) need eight
//   different chunks among the rows of equal parity, column reads (four rows
//   4 i .. 4 i + 3, 64 bytes each) 64 bytes between rows 4 i and 4 i + 2.
//   swz(r) = bits 1..3 of r with bit 1 of r moved to bit 2, where it flips 64
//   bytes, satisfies both.
//   DH 128: rows are 768 bytes, a multiple of the window: 16 different chunks
//   for 16 rows, and 64 bytes apart for four consecutive rows:
//   swz(r) = bits 0..3 of r with the low two moved to bits 2 and 3.
#pragma once

#include "vedic_flash_attn.hpp"
#include "vedic_gemm_f16.hpp"
#include "vedic_split.hpp"

namespace vedic {

template <int DH>
__device__ __forceinline__ int fs_swz(int r) {
    if constexpr (DH == 64) return (((r >> 1) & 1) << 2) | ((r >> 2) & 3);
    else return ((r & 3) << 2) | ((r >> 2) & 3);
}
template <int DH>
constexpr int fs_block_bytes() {
    return 32 * 6 * DH;
}

// One block's values in the registers of NT threads: unit u = i NT + tid is
// the eight values of chunk u % (DH / 8) of row u / (DH / 8).
template <int DH, int NT>
struct FsStage {
    static constexpr int CPR = DH / 8;
    static constexpr int U = 32 * CPR / NT;
    static_assert(32 * CPR % NT == 0, "units divide among the threads");
    float v[U][8];

    // Rows row0 .. of X; those at or past `rows` (from row0) load as zeros.
    __device__ __forceinline__ void load(const float* X, int row0, int rows, int tid) {
        const __amdgpu_buffer_rsrc_t rs = buffer_rsrc(X + (rows > 0 ? (int64_t)row0 * DH : 0));
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int u = i * NT + tid, row = u / CPR;
            const uint32_t off = row < rows ? (uint32_t)(u * 32) : kOob;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const float4_t w = __builtin_bit_cast(
                    float4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(off == kOob ? kOob : off + 16 * q), 0, 0));
#pragma unroll
                for (int e = 0; e < 4; ++e) v[i][4 * q + e] = w[e];
            }
        }
    }
    // Their parts, scaled by `scale`, into the block at `lds`.
    __device__ __forceinline__ void commit(char* lds, float scale, int tid) const {
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int u = i * NT + tid, row = u / CPR, c = u % CPR;
            const SplitFrag f = split8(v[i], scale);
            char* dst = lds + row * 6 * DH + ((c ^ fs_swz<DH>(row)) << 4);
#pragma unroll
            for (int p = 0; p < 3; ++p) *reinterpret_cast<bf16x8_t*>(dst + p * 2 * DH) = f.p[p];
        }
    }
};

// A lane's read positions in a block.  The steps j and d and the halves t of a
// column read only flip chunk bits, which no row offset touches (rows are
// multiples of 128 and 256 bytes), so every other address is one XOR away.
template <int DH>
struct FsAddr {
    uint32_t row;  // row l32, chunk h
    uint32_t col;  // row 4 h + (lane % 16) / 4, the lane's 8 bytes of columns 0 .. 31
    __device__ __forceinline__ explicit FsAddr(int lane) {
        const int l32 = lane & 31, h = lane >> 5, s = lane & 15;
        row = (uint32_t)(l32 * 6 * DH + ((h ^ fs_swz<DH>(l32)) << 4));
        const int r = 4 * h + (s >> 2), c = 2 * ((lane >> 4) & 1) + ((s & 3) >> 1);
        col = (uint32_t)(r * 6 * DH + ((c ^ fs_swz<DH>(r)) << 4) + 8 * (s & 1));
    }
    // Keeps the derived addresses from living across a whole loop.
    __device__ __forceinline__ void refresh() { asm volatile("" : "+v"(row), "+v"(col)); }
};

// Operand of a product over DH: row l32, values 16 j + 8 h .. + 7.
template <int DH>
__device__ __forceinline__ SplitFrag fs_row(const char* blk, const FsAddr<DH>& ad, int j) {
    const char* p = blk + (ad.row ^ (uint32_t)(j << 5));
    SplitFrag f;
#pragma unroll
    for (int q = 0; q < 3; ++q) f.p[q] = *reinterpret_cast<const bf16x8_t*>(p + q * 2 * DH);
    return f;
}

// Operand of a product over the block's rows, in the order the 32 x 32
// accumulator holds them (so that an accumulator can be the other operand as
// it is): column 32 d + l32, element e of lane half h is row
// 16 j + 8 (e / 4) + 4 h + e % 4.
template <int DH>
__device__ __forceinline__ SplitFrag fs_col(const char* blk, const FsAddr<DH>& ad, int d, int j) {
    SplitFrag f;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
        union {
            short4_t q[2];
            bf16x8_t h;
        } u;
#pragma unroll
        for (int t = 0; t < 2; ++t)
            u.q[t] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (lds_short4_t*)(blk + (ad.col ^ (uint32_t)((d << 6) | (t << 5))) + (16 * j + 8 * t) * 6 * DH + p * 2 * DH));
        f.p[p] = u.h;
    }
    return f;
}

// Rows (query or key) q0 + l32 of X as operands over DH, scaled by `scale`
// before the split; zeros past seq.
template <int DH>
__device__ __forceinline__ void fs_load_rows(SplitFrag (&f)[DH / 16], const float* X, int row, int seq, float scale,
                                             int lane) {
    const __amdgpu_buffer_rsrc_t rs = buffer_rsrc(X);
    const uint32_t off = row < seq ? (uint32_t)(row * DH * 4 + (lane >> 5) * 32) : kOob;
#pragma unroll
    for (int j = 0; j < DH / 16; ++j) {
        float w[8];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const float4_t t = __builtin_bit_cast(
                float4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(off == kOob ? kOob : off + 64 * j + 16 * q), 0, 0));
#pragma unroll
            for (int e = 0; e < 4; ++e) w[4 * q + e] = t[e];
        }
        f[j] = split8(w, scale);
    }
}

// The parts of accumulator registers 8 j .. 8 j + 7, times `scale`: the operand
// that meets fs_col(.., j, ..).
__device__ __forceinline__ SplitFrag fs_acc(const float16_t& s, int j, float scale) {
    float w[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) w[e] = s[8 * j + e];
    return split8(w, scale);
}

}  // namespace vedic
