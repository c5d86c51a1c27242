// mfa_bwd_common.h -- definitions shared by the 16-bit (mfa_bwd.hip) and fp32
// (mfa_bwd32.hip) backward kernels: the kernel argument block and the fp32
// kernels' table.
#pragma once

#include "mfa_common.h"

// Kernels of the fp32 backward (mfa_bwd32.hip), each a void(*)(BArgs).
constexpr int kB32Rows = 32;  // query rows per dQ workgroup
constexpr int kB32Keys = 32;  // keys per dK/dV workgroup
struct Bwd32Kernels {
    void *dkdv, *dq;
};
// Two workgroups of these kernels share a CU up to this padded head dim, one above.
constexpr int kB32PairDim = 64;
// dp: head dim padded to 32/64/96/128; bias: soft-cap or ALiBi
__attribute__((visibility("hidden"))) Bwd32Kernels mfa_bwd32_kernels(int dp, bool bias);

namespace {

constexpr int kBThreads = 256;  // 4 wavefronts

struct BArgs {
    KArgs f;  // forward arguments: q, k, v, o, strides, shapes, masks, lse (input)
    const char* dout;
    int64_t dob, dos, doh;
    char* dq;
    int64_t dqb, dqs, dqh;
    char* dk;
    int64_t dkb, dks, dkh;
    char* dv;
    int64_t dvb, dvs, dvh;
    float* dsum;       // [B*Hq][Lq] rowsum(dO * O) - dlse
    const float* dlse; // gradient of lse (softmax_lse layout), or NULL
    int32_t grad_f32;  // dq/dk/dv written as fp32
    int32_t T;         // tiles per unit (dK/dV: key tiles; dQ: query tiles)
    int32_t fold;      // fp32 kernels: tile slots from here on run in reverse order (0: off)
    int32_t Ukv;       // (sequence, K/V head) units = B * Hkv
    // grouped-query heads split over dK/dV workgroups: G groups of R/G query
    // heads each; G > 1 writes fp32 partials ws_dk/ws_dv [G][B*Hkv][Lk][DP]
    // that mfa_bwd_dkdv_sum_kernel adds in group order
    int32_t G;
    int32_t ws_ld;  // DP
    float* ws_dk;
    float* ws_dv;
};

// exp2-domain lse of a row for P = exp2(s*c - lse2): lse*log2(e), and +inf for
// a row with no valid key (so its P is 0).
__device__ __forceinline__ float lse2_of(float lse) { return lse == -INFINITY ? INFINITY : lse * kLog2e; }

}  // namespace
