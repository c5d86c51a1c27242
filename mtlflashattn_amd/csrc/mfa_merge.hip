// mfa_merge.hip -- merge of attention partials over disjoint key sets
// (mfa_merge in include/mfa.h): out = sum_i w_i out_i with
// w_i = exp(lse_i - lse), lse = ln(sum_i exp(lse_i)).
//
// Bound by memory: every partial is read once and the result written once.
// One workgroup takes 16 positions x 4 heads: 64 threads form the weights of
// those 64 rows from the parts' lse (16 consecutive floats per head) and put
// them in LDS, then all 256 stream the rows in 16-byte chunks, every part's
// chunk of a thread in flight at once.  Measured on four bf16 parts of
// B=1 L=4096 H=16 D=128 (85 MB): 21.8 us per call, 3.9 TB/s (a large copy
// reaches 5.1); as separate elementwise passes (stack, logsumexp, one cast /
// multiply / add per part over fp32 temporaries) the same call was 50 launches
// and 238 us.
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include "mfa.h"
#include "mfa_common.h"

namespace {

constexpr int kMThreads = 256;
constexpr int kMPos = 16, kMHeads = 4, kMRows = kMPos * kMHeads;

struct MArgs {
    const char* o[MFA_MERGE_MAX_PARTS];
    const float* lse[MFA_MERGE_MAX_PARTS];
    int64_t ob[MFA_MERGE_MAX_PARTS], os[MFA_MERGE_MAX_PARTS], oh[MFA_MERGE_MAX_PARTS];  // elements
    int64_t lb[MFA_MERGE_MAX_PARTS], lh[MFA_MERGE_MAX_PARTS], ls[MFA_MERGE_MAX_PARTS];
    char* out;       // [B, L, H, D] contiguous
    float* lse_out;  // [B, H, L] contiguous
    int32_t n, L, H, D;
    int32_t lt, ht;  // position and head tiles
};

// DT: MFA_DTYPE_*; a 16-byte chunk as floats and back
template <int DT>
struct Chunk {
    static constexpr int ES = DT == MFA_DTYPE_F32 ? 4 : 2;
    static constexpr int N = 16 / ES;
    __device__ static __forceinline__ void load(const u32x4_t& w, float (&x)[N]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t v = w[i];
            if constexpr (DT == MFA_DTYPE_F32) {
                x[i] = __uint_as_float(v);
            } else if constexpr (DT == MFA_DTYPE_BF16) {
                x[2 * i] = __uint_as_float(v << 16);
                x[2 * i + 1] = __uint_as_float(v & 0xffff0000u);
            } else {
                x[2 * i] = (float)__builtin_bit_cast(_Float16, (uint16_t)(v & 0xffffu));
                x[2 * i + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(v >> 16));
            }
        }
    }
    __device__ static __forceinline__ u32x4_t pack(const float (&x)[N]) {
        u32x4_t w;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (DT == MFA_DTYPE_F32) {
                w[i] = __float_as_uint(x[i]);
            } else if constexpr (DT == MFA_DTYPE_BF16) {
                typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 v2;
                const v2 p = {(__bf16)x[2 * i], (__bf16)x[2 * i + 1]};
                w[i] = __builtin_bit_cast(uint32_t, p);
            } else {
                typedef __attribute__((__vector_size__(2 * sizeof(_Float16)))) _Float16 v2;
                const v2 p = {(_Float16)x[2 * i], (_Float16)x[2 * i + 1]};
                w[i] = __builtin_bit_cast(uint32_t, p);
            }
        }
        return w;
    }
};

template <int DT>
__global__ void __launch_bounds__(kMThreads) mfa_merge_kernel(MArgs a) {
    typedef Chunk<DT> C;
    __shared__ float w_s[MFA_MERGE_MAX_PARTS][kMRows];  // row = head * kMPos + position
    const int tid = threadIdx.x;
    const int ltile = blockIdx.x % a.lt, bh = blockIdx.x / a.lt;
    const int htile = bh % a.ht, b = bh / a.ht;
    const int l0 = ltile * kMPos, h0 = htile * kMHeads;
    if (tid < kMRows) {
        const int l = l0 + (tid % kMPos), h = h0 + tid / kMPos;
        if (l < a.L && h < a.H) {
            // (the arithmetic of a log-sum-exp over the parts: NaN spreads, a
            // +inf or all -inf row gets that lse and weights of 0)
            float m = -INFINITY;
            for (int i = 0; i < a.n; ++i) {
                const float x = a.lse[i][b * a.lb[i] + h * a.lh[i] + l * a.ls[i]];
                w_s[i][tid] = x;
                m = fmax_nn(m, x);
            }
            const float ref = __builtin_isinf(m) ? 0.f : m;
            float sum = 0.f;
            for (int i = 0; i < a.n; ++i) sum += expf(w_s[i][tid] - ref);
            const float lse = logf(sum) + ref;
            const bool off = __builtin_isinf(lse);
            for (int i = 0; i < a.n; ++i) w_s[i][tid] = off ? 0.f : expf(w_s[i][tid] - lse);
            a.lse_out[((int64_t)b * a.H + h) * a.L + l] = lse;
        }
    }
    __syncthreads();
    const int cpr = a.D / C::N;  // chunks per row
    const int nh = min(kMHeads, a.H - h0), nl = min(kMPos, a.L - l0);
    const int total = nl * nh * cpr;
    for (int cc = tid; cc < total; cc += kMThreads) {
        const int row = cc / cpr, col = (cc - row * cpr) * C::N;
        const int pl = row / nh, hh = row - pl * nh;  // heads run fastest, as in memory
        const int64_t l = l0 + pl, h = h0 + hh;
        const int wr = hh * kMPos + pl;
        float acc[C::N];
        auto add = [&](int i, const u32x4_t& v) {
            float x[C::N];
            C::load(v, x);
            const float w = w_s[i][wr];
#pragma unroll
            for (int e = 0; e < C::N; ++e) acc[e] = i == 0 ? w * x[e] : fmaf(w, x[e], acc[e]);
        };
        auto src = [&](int i) {
            return reinterpret_cast<const u32x4_t*>(a.o[i] + (b * a.ob[i] + l * a.os[i] + h * a.oh[i] + col) * C::ES);
        };
        int i = 0;
        for (; i + 4 <= a.n; i += 4) {
            u32x4_t v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = *src(i + k);
#pragma unroll
            for (int k = 0; k < 4; ++k) add(i + k, v[k]);
        }
        for (; i < a.n; ++i) add(i, *src(i));
        store_stream(reinterpret_cast<u32x4_t*>(a.out + ((((int64_t)b * a.L + l) * a.H + h) * a.D + col) * C::ES),
                     C::pack(acc));
    }
}

int merr(int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(mfa_error_buffer(), 512, fmt, ap);
    va_end(ap);
    return code;
}

}  // namespace

extern "C" {

int mfa_merge_params_size(void) { return (int)sizeof(mfa_merge_params); }

int mfa_merge(const mfa_merge_params* p, void* stream) {
    mfa_error_buffer()[0] = 0;
    if (!p) return merr(MFA_ERR_INVALID, "mfa_merge: params is NULL");
    if (p->dtype != MFA_DTYPE_F16 && p->dtype != MFA_DTYPE_BF16 && p->dtype != MFA_DTYPE_F32)
        return merr(MFA_ERR_INVALID, "mfa_merge: unknown dtype %d", p->dtype);
    if (p->parts < 1 || p->parts > MFA_MERGE_MAX_PARTS)
        return merr(MFA_ERR_INVALID, "mfa_merge: %d parts outside [1, %d]", p->parts, MFA_MERGE_MAX_PARTS);
    if (p->batch < 0 || p->seqlen < 0 || p->heads < 0 || p->head_dim < 0)
        return merr(MFA_ERR_INVALID, "mfa_merge: negative size");
    if (p->batch == 0 || p->seqlen == 0 || p->heads == 0 || p->head_dim == 0) return MFA_OK;
    const int al = p->dtype == MFA_DTYPE_F32 ? 4 : 8;  // elements per 16 bytes
    if (p->head_dim % al) return merr(MFA_ERR_UNSUPPORTED, "mfa_merge: head_dim %d is not a multiple of %d", p->head_dim, al);
    auto bad = [](const void* x, uintptr_t a) { return !x || (reinterpret_cast<uintptr_t>(x) & (a - 1)); };
    if (bad(p->out, 16) || bad(p->lse_out, 4))
        return merr(MFA_ERR_INVALID, "mfa_merge: out (16-byte aligned) and lse_out are required");
    MArgs a;
    memset(&a, 0, sizeof(a));
    for (int i = 0; i < p->parts; ++i) {
        const mfa_merge_part& q = p->part[i];
        if (bad(q.o, 16) || bad(q.lse, 4))
            return merr(MFA_ERR_INVALID, "mfa_merge: part %d: o (16-byte aligned) and lse are required", i);
        if (q.o_batch_stride % al || q.o_seq_stride % al || q.o_head_stride % al)
            return merr(MFA_ERR_INVALID, "mfa_merge: part %d: o strides must be multiples of %d elements", i, al);
        a.o[i] = static_cast<const char*>(q.o);
        a.lse[i] = q.lse;
        a.ob[i] = q.o_batch_stride; a.os[i] = q.o_seq_stride; a.oh[i] = q.o_head_stride;
        a.lb[i] = q.lse_batch_stride; a.lh[i] = q.lse_head_stride; a.ls[i] = q.lse_seq_stride;
    }
    a.out = static_cast<char*>(p->out);
    a.lse_out = p->lse_out;
    a.n = p->parts;
    a.L = p->seqlen; a.H = p->heads; a.D = p->head_dim;
    a.lt = (p->seqlen + kMPos - 1) / kMPos;
    a.ht = (p->heads + kMHeads - 1) / kMHeads;
    const int64_t grid = (int64_t)p->batch * a.ht;  // (bounded before the next product)
    if (grid > 0x7fffffffLL || grid * a.lt > 0x7fffffffLL || (int64_t)kMRows * p->head_dim > 0x7fffffffLL)
        return merr(MFA_ERR_INVALID, "mfa_merge: problem too large");
    const auto fn = p->dtype == MFA_DTYPE_F32    ? mfa_merge_kernel<MFA_DTYPE_F32>
                    : p->dtype == MFA_DTYPE_BF16 ? mfa_merge_kernel<MFA_DTYPE_BF16>
                                                 : mfa_merge_kernel<MFA_DTYPE_F16>;
    hipLaunchKernelGGL(fn, dim3((unsigned)(grid * a.lt)), dim3(kMThreads), 0, static_cast<hipStream_t>(stream), a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return merr(MFA_ERR_LAUNCH, "mfa_merge: launch failed: %s", hipGetErrorString(e));
    return MFA_OK;
}

}  // extern "C"
