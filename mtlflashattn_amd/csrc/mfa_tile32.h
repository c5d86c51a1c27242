// mfa_tile32.h -- fp32 tiles of one wavefront and their products on the fp32
// matrix cores (v_mfma_f32_32x32x2_f32), shared by the fp32 forward
// (mfa_fwd.hip) and backward (mfa_bwd32.hip).
//
// In the 32x32x2 MFMA lane (half, x) supplies row or column x of the operands
// at k = half, and holds column x of the accumulator, register r at row
// acc_row(r) + 4 * half.  So register r of an accumulator is, as it stands, the
// B operand of an MFMA over the two rows acc_row(r) and acc_row(r) + 4.
#pragma once

#include "mfa_common.h"

namespace {

__device__ __forceinline__ f32x16_t mfma32(float x, float y, const f32x16_t& acc) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(x, y, acc, 0, 0, 0);
}

// A 32-row tile of one wavefront in LDS: rows of DP floats, unpadded (direct
// loads write lane i at 16 * i), with chunk c (16 bytes) of row r in slot
// c ^ swz(r).  The swizzle spreads 16 consecutive rows' equal chunks over the
// 16 slots of a 256-byte line, so the row reads (one row per lane, 16 bytes)
// are free of bank conflicts, and the column reads (32 consecutive floats of
// one row per half-wavefront) always are.
template <int DP>
struct Tile {
    static constexpr int CPR = DP / 4;         // chunks per row
    static constexpr int N = 32 * CPR / 64;    // loads of 64 x 16 bytes per tile
    static constexpr int FLOATS = 32 * DP;
    static constexpr bool kWide = CPR % 16 == 0;  // rows are whole 256-byte lines
    __device__ static __forceinline__ int swz(int r) { return kWide ? r & 15 : (r >> 1) & 7; }

    // Issue the loads of rows [0, rows) of a [rows, D] matrix of row stride
    // `st` floats; rows and columns past the matrix read as 0.  `wide`: 32
    // rows span 2 GiB or more, beyond a buffer resource's 32-bit offsets
    // (plain loads then, complete when the call returns).
    __device__ static __forceinline__ void load(float* dst, const float* src, int64_t st, int rows, int D, int lane,
                                                bool wide) {
        int l = lane;
        pin(l);  // (the offsets are formed here, not kept in registers through the walk)
        if (!wide) {
            const uint32_t bytes =
                (uint32_t)__builtin_amdgcn_readfirstlane(rows > 0 ? (int)(((rows - 1) * st + D) * 4) : 0);
            const uint32_t st32 = (uint32_t)st;
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const int cc = 64 * i + l, row = cc / CPR, col = ((cc % CPR) ^ swz(row)) * 4;
                const uint32_t off = (row < rows && col < D) ? (row * st32 + col) * 4 : 0x80000000u;
                lds_load16(reinterpret_cast<uint64_t>(src), bytes, reinterpret_cast<uint16_t*>(dst + 256 * i), off);
            }
        } else {
#pragma unroll 1
            for (int i = 0; i < N; ++i) {
                const int cc = 64 * i + l, row = cc / CPR, col = ((cc % CPR) ^ swz(row)) * 4;
                float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
                if (row < rows && col < D) v = *reinterpret_cast<const float4*>(src + row * st + col);
                *reinterpret_cast<float4*>(dst + cc * 4) = v;
            }
        }
    }

    // acc += T B over the head dim: A operand = rows of the tile, B operand
    // `y` with k-slot `half` of step s at d = s + half * DP/2.
    __device__ static __forceinline__ void rows_product(const float* t, const float (&y)[DP / 2], int l32, int half,
                                                        f32x16_t& acc) {
        int x = l32;
        pin(x);
        const float* row = t + x * DP;
        const int f = swz(x), c0 = half * (DP / 8);
#pragma unroll
        for (int s = 0; s < DP / 8; ++s) {
            const float4 w = *reinterpret_cast<const float4*>(row + (((c0 + s) ^ f) << 2));
            acc = mfma32(w.x, y[4 * s], acc);
            acc = mfma32(w.y, y[4 * s + 1], acc);
            acc = mfma32(w.z, y[4 * s + 2], acc);
            acc = mfma32(w.w, y[4 * s + 3], acc);
        }
    }

    // Lane offsets of the column reads (row 4 * half, this lane's column of a
    // 32-column block), one per class of rows with the same lane-dependent swizzle.
    __device__ static __forceinline__ void col_offsets(int (&off)[4], int l32, int half) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int f = kWide ? 4 * half + j : 4 * (j >> 1) + 2 * half + (j & 1);
            off[j] = 4 * half * DP + (((l32 >> 2) ^ f) << 2) + (l32 & 3);
        }
    }
    // acc[db] += T^T B: A operand = columns 32*db.. of the tile's rows
    // acc_row(r) + 4 * half, B operand = register r of p.
    template <int DB>
    __device__ static __forceinline__ void cols_product(const float* t, const int (&off)[4], const f32x16_t& p,
                                                        f32x16_t (&acc)[DB]) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int j = kWide ? (r & 3) : 2 * ((r >> 2) & 1) + ((r >> 1) & 1);
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                const int cb = kWide ? db ^ ((r >> 2) & 1) : db;
                acc[db] = mfma32(t[off[j] + acc_row(r) * DP + 32 * cb], p[r], acc[db]);
            }
        }
    }

    // A transposed accumulator (lane = row, registers = columns) into the tile.
    template <int DB>
    __device__ static __forceinline__ void put(float* t, const f32x16_t (&acc)[DB], int l32, int half) {
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *reinterpret_cast<float4*>(t + l32 * DP + (((8 * db + 2 * g + half) ^ swz(l32)) << 2)) =
                    make_float4(acc[db][4 * g], acc[db][4 * g + 1], acc[db][4 * g + 2], acc[db][4 * g + 3]);
    }
    // Sum of the four wavefronts' tiles (`step` floats apart), in order, to
    // rows [0, rows) of a [rows, D] matrix, all threads of the workgroup.
    __device__ static __forceinline__ void sum4(const float* t, int step, float* dst, int64_t st, int rows, int D,
                                                int tid) {
#pragma unroll 2
        for (int cc = tid; cc < 32 * CPR; cc += 256) {
            const int row = cc / CPR, col = ((cc % CPR) ^ swz(row)) * 4;
            if (row >= rows || col >= D) continue;
            float4 s = *reinterpret_cast<const float4*>(t + cc * 4);
#pragma unroll
            for (int w = 1; w < 4; ++w) {
                const float4 x = *reinterpret_cast<const float4*>(t + w * step + cc * 4);
                s.x += x.x;
                s.y += x.y;
                s.z += x.z;
                s.w += x.w;
            }
            *reinterpret_cast<float4*>(dst + row * st + col) = s;
        }
    }
};

// This lane's row of an [L, D] matrix as the B operand of rows_product: k-slot
// `half` of step s holds d = s + half * DP/2 (0 past the matrix).
template <int DP>
__device__ __forceinline__ void row_operand(float (&y)[DP / 2], const float* src, bool in, int D, int half) {
#pragma unroll
    for (int s = 0; s < DP / 2; s += 4) {
        const int d = s + half * (DP / 2);
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (in && d < D) v = *reinterpret_cast<const float4*>(src + d);
        y[s] = v.x;
        y[s + 1] = v.y;
        y[s + 2] = v.z;
        y[s + 3] = v.w;
    }
}

}  // namespace
