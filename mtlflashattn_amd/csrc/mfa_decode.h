// mfa_decode.h -- what the planner (mfa_fwd.hip) and the single-row kernels
// (mfa_decode.hip) share: the chunking of a sequence's keys, the argument
// block and the kernel table.
#pragma once

#include "mfa_common.h"

// Keys per chunk of a single-row sequence of Lk keys.  The softmax of a row is
// formed chunk by chunk and the chunks' results are added in order, so the
// chunk length is part of the result's rounding: it depends on the sequence's
// own key count alone, never on the batch, the launch shape or a caller's
// split.  256 keys (two 32-key blocks per wavefront) give a few thousand keys
// enough workgroups to fill the chip; longer sequences take longer chunks, so
// that no sequence below 128K keys has more than 64 partial results to merge.
__host__ __device__ inline int decode_chunk(int Lk) {
    return Lk <= 16384 ? 256 : Lk <= 32768 ? 512 : Lk <= 65536 ? 1024 : 2048;
}
__host__ __device__ inline int decode_chunks(int Lk) {
    const int c = decode_chunk(Lk);
    return Lk > 0 ? (Lk + c - 1) / c : 1;
}
// most chunks of any sequence of at most Lk keys
__host__ inline int decode_chunks_max(int Lk) {
    const int n = decode_chunks(Lk);
    return Lk > 16384 && n < 64 ? 64 : n;
}

constexpr int kDecodeRows = 16;    // query heads of a K/V head per workgroup
constexpr int kDecodeThreads = 256;

namespace {

struct DArgs {
    KArgs f;         // tensors, strides, shapes, masks (f.Lk the longest sequence; every computed row is a single one)
    int32_t R;       // query heads per K/V head
    int32_t nr;      // min(R, kDecodeRows): heads of a full tile
    int32_t rt;      // tiles of kDecodeRows heads per K/V head
    int32_t units;   // (sequence, K/V head, tile)
    int32_t nsplit;  // workgroups per unit: workgroup (split, unit) takes chunks split * group .. + group - 1
    int32_t group;
    int32_t nt;      // K/V loads non-temporal
    int32_t bias;    // soft-cap, ALiBi or a scale that is not positive
    int32_t ws_ld;   // floats per partial row
    float* ws_o;     // [chunk][units * nr][ws_ld] chunk sums of p v
    float* ws_ml;    // [chunk][units * nr][2] exponent reference, sum of p
};

}  // namespace

struct DecodeKernels {
    void *attend, *merge;  // void(*)(DArgs)
    int lds;
};
// dp: head dim padded to 32/64/96/128
__attribute__((visibility("hidden"))) DecodeKernels mfa_decode_kernels(int dp, bool bf16, bool paged);
