// mfa_decode.hip -- attention of single query rows (decode): sequences whose
// query is one token, bf16 / fp16.
//
// Bound by the K/V stream (HBM) when the batch is large and by latency and
// empty compute units when it is small, so the kernel is built around the
// loads:
//  * The query heads of a K/V head are the columns of one 16-column MFMA
//    (v_mfma_f32_16x16x32), so K and V are read once for up to 16 heads.
//  * A sequence's keys are cut into chunks (decode_chunk).  One workgroup takes
//    a chunk: its four wavefronts take every fourth 32-key block, each loading
//    straight to its own LDS tiles (no barrier), and hold a softmax state of
//    their own; the four are added at the chunk's end.
//  * A workgroup walks as many consecutive chunks as keep the chip full, its
//    loads running on across the chunk ends: all of its unit's with many units,
//    one with few.  Where it has not all of them, each chunk's sums go to a
//    workspace and a second kernel adds them.
// Either way gives the same bits.  Every exponent reference is an integer (the
// ceiling of the row maximum in the exp2 domain), so rescaling is a
// multiplication by a power of two, exact, and the sum over wavefronts and
// chunks in their order does not depend on which reference was current.  (Terms
// below 2^-126 of the row's largest weight may differ.)
//  * Probabilities are carried as two 16-bit terms, hi = round16(p) and
//    lo = round16(p - hi), both fed to the PV MFMA: a row over thousands of
//    near-equal weights averages V, and one 16-bit rounding of every weight
//    would be visible against its small result.  Row sums are fp32.
#include <math.h>
#include <stdint.h>

#include "mfa.h"
#include "mfa_decode.h"

namespace {

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;
constexpr float kDLn2 = 0.6931471805599453f;

// max over the four 16-lane groups (each lane of a group is one query column)
__device__ __forceinline__ float max_groups(float x) {
    auto a = __builtin_amdgcn_permlane16_swap(__float_as_int(x), __float_as_int(x), false, false);
    return max_halves(fmax_nn(__int_as_float(a[0]), __int_as_float(a[1])));
}
__device__ __forceinline__ float sum_groups(float x) {
    auto a = __builtin_amdgcn_permlane16_swap(__float_as_int(x), __float_as_int(x), false, false);
    return sum_halves(__int_as_float(a[0]) + __int_as_float(a[1]));
}

template <bool IS_BF16>
struct Ops16 {
    typedef typename std::conditional<IS_BF16, bf16x8_t, f16x8_t>::type op_t;
    __device__ static __forceinline__ f32x4_t mfma(const op_t& x, const op_t& y, const f32x4_t& acc) {
        if constexpr (IS_BF16)
            return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, acc, 0, 0, 0);
        else
            return __builtin_amdgcn_mfma_f32_16x16x32_f16(x, y, acc, 0, 0, 0);
    }
    // two floats as hi = round16 and lo = round16(x - hi), packed
    __device__ static __forceinline__ void split(float x, float y, uint32_t& hi, uint32_t& lo) {
        if constexpr (IS_BF16) {
            typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 v2;
            const v2 h = {(__bf16)x, (__bf16)y};
            hi = __builtin_bit_cast(uint32_t, h);
            const v2 l = {(__bf16)(x - __uint_as_float(hi << 16)), (__bf16)(y - __uint_as_float(hi & 0xffff0000u))};
            lo = __builtin_bit_cast(uint32_t, l);
        } else {
            typedef __attribute__((__vector_size__(2 * sizeof(_Float16)))) _Float16 v2;
            const v2 h = {(_Float16)x, (_Float16)y};
            hi = __builtin_bit_cast(uint32_t, h);
            const v2 l = {(_Float16)(x - (float)h[0]), (_Float16)(y - (float)h[1])};
            lo = __builtin_bit_cast(uint32_t, l);
        }
    }
    // two ds_read_b64_tr_b16: in each 16-lane group lane i addresses 4
    // elements of row i/4 and receives element i of rows 0..3
    __device__ static __forceinline__ op_t load_tr(const uint16_t* p0, const uint16_t* p1) {
        if constexpr (IS_BF16) {
            typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 v4;
            typedef __attribute__((address_space(3))) v4* lp;
            return __builtin_shufflevector(__builtin_amdgcn_ds_read_tr16_b64_v4bf16((lp)(p0)),
                                           __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lp)(p1)), 0, 1, 2, 3, 4, 5, 6, 7);
        } else {
            typedef __attribute__((__vector_size__(4 * sizeof(__fp16)))) __fp16 v4h;
            typedef __attribute__((__vector_size__(4 * sizeof(_Float16)))) _Float16 v4;
            typedef __attribute__((address_space(3))) v4h* lp;
            const v4 lo = __builtin_bit_cast(v4, __builtin_amdgcn_ds_read_tr16_b64_v4f16((lp)(p0)));
            const v4 hi = __builtin_bit_cast(v4, __builtin_amdgcn_ds_read_tr16_b64_v4f16((lp)(p1)));
            return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        }
    }
};

// One result row's D elements at d..d+3 (o = sum of p v, l = sum of p).
template <bool IS_BF16>
__device__ __forceinline__ void store4(const KArgs& f, char* row, int d, const f32x4_t& o, float l) {
    f32x4_t x;
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = l > 0.f ? o[i] / l : o[i];  // (l = 0: no key, o = 0; NaN stays NaN)
    if (f.out_f32) {
        store_stream(reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(row) + d), x);
    } else if constexpr (IS_BF16) {
        typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 v4;
        store_stream(reinterpret_cast<v4*>(reinterpret_cast<__bf16*>(row) + d),
                     v4{(__bf16)x[0], (__bf16)x[1], (__bf16)x[2], (__bf16)x[3]});
    } else {
        typedef __attribute__((__vector_size__(4 * sizeof(_Float16)))) _Float16 v4;
        store_stream(reinterpret_cast<v4*>(reinterpret_cast<_Float16*>(row) + d),
                     v4{(_Float16)x[0], (_Float16)x[1], (_Float16)x[2], (_Float16)x[3]});
    }
}

// The unit (sequence, K/V head, tile of heads) of a workgroup.
struct Unit {
    int b, hkv, h0, nr;  // first query head and number of heads
    int tok;             // varlen: the sequence's token (0 dense)
    int k_start, Lq, Lk;
};
__device__ __forceinline__ Unit unit_of(const DArgs& a, int unit) {
    const KArgs& f = a.f;
    Unit u;
    const int g = unit / a.rt, t = unit - g * a.rt;
    u.b = g / f.Hkv;
    u.hkv = g - u.b * f.Hkv;
    u.h0 = u.hkv * a.R + t * kDecodeRows;
    u.nr = min(kDecodeRows, a.R - t * kDecodeRows);
    u.tok = u.k_start = 0;
    u.Lq = 1;
    u.Lk = f.Lk;
    if (f.cu_q) {
        u.tok = f.cu_q[u.b];
        u.Lq = f.cu_q[u.b + 1] - u.tok;
        u.k_start = f.cu_k[u.b];
        u.Lk = f.cu_k[u.b + 1] - u.k_start;
    }
    return u;
}
__device__ __forceinline__ char* out_row(const KArgs& f, const Unit& u, int r) {
    const int64_t off = (f.cu_q ? u.tok * f.os : u.b * f.ob) + (int64_t)(u.h0 + r) * f.oh;
    return f.o + off * (f.out_f32 ? 4 : 2);
}
__device__ __forceinline__ void store_lse(const KArgs& f, const Unit& u, int r, float m, float l) {
    if (!f.lse) return;
    float* p = f.lse + (f.cu_q ? (int64_t)u.tok : u.b * f.lse_b) + (int64_t)(u.h0 + r) * f.lse_h;
    *p = m == -INFINITY ? -INFINITY : (m + __builtin_amdgcn_logf(l)) * kDLn2;
}

// One K and one V tile of LDS per wavefront: the next K loads run behind the
// softmax and PV, the next V behind QK.  Two of each, loading two steps ahead,
// measured slower wherever bandwidth counts (with plain loads, 24 sequences to
// 4096 keys, Hq=32 Hkv=8 D=128, two chunks per workgroup: 66.6 against 56.0 us;
// B=64 Lk=4096 the same: 187.8 and 186.6): with 64 KB at head dim 128 two workgroups share a CU,
// and one streams while the other starts, merges or ends.
template <int DP, bool IS_BF16, bool PAGED>
__global__ void __launch_bounds__(kDecodeThreads) mfa_fwd16x_kernel(DArgs a) {
    typedef Ops16<IS_BF16> O;
    typedef typename O::op_t op_t;
    constexpr int CPR = DP / 8;        // 16-byte chunks per row
    constexpr int NL = 32 * CPR / 64;  // loads of 64 x 16 bytes per 32-key tile
    constexpr int TILE = 32 * DP;      // elements of a K or V tile
    constexpr int ITEMS = (kDecodeRows * (DP / 4) + kDecodeThreads - 1) / kDecodeThreads;  // 4-element pieces per thread
    static_assert(kDecodeRows * DP * 4 <= TILE * 2, "a V tile holds a wavefront's sums");
    __shared__ __attribute__((aligned(16))) uint16_t smem[4][2][TILE];  // [wavefront][K, V]
    __shared__ float m_s[4][kDecodeRows], l_s[4][kDecodeRows];

    const KArgs& f = a.f;
    const int split = blockIdx.x / a.units, unit = blockIdx.x - split * a.units;
    const Unit u = unit_of(a, unit);
    if (u.Lq != 1) return;  // (varlen: empty sequences, and longer ones, which are another launch's)
    const int Lk = u.Lk, D = f.D;
    const int chunk = decode_chunk(Lk), nchunks = decode_chunks(Lk);
    const int c_first = split * a.group;  // the chunks of this workgroup: `group` from here on
    if (c_first >= nchunks) return;
    const bool whole = a.group >= nchunks;  // all of the unit's: the result is stored here
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, grp = lane >> 4;

    // the row's valid keys (the query is the last position), the chunks walked
    const int center = Lk - 1, lo = key_lo(f, center), hi = key_hi(f, center, Lk);
    const int c_beg = whole ? lo / chunk : c_first, c_end = min(c_first + a.group, nchunks);
    // 32-key blocks per wavefront and chunk: the same number of steps for every
    // chunk (the last may be short), so the stages alternate alike everywhere
    const int spc = chunk / 128;
    const int steps = (c_end - c_beg) * spc;

    // K/V of this head
    const char* kbase = f.k + ((PAGED ? 0 : f.cu_k ? (int64_t)u.k_start * f.ks : u.b * f.kb) + u.hkv * f.kh) * 2;
    const char* vbase = f.v + ((PAGED ? 0 : f.cu_k ? (int64_t)u.k_start * f.vs : u.b * f.vb) + u.hkv * f.vh) * 2;
    const int32_t* bt = PAGED ? f.bt + u.b * f.bt_b : nullptr;

    // Tiles in LDS: unpadded rows (a direct load writes lane i at 16 * i), chunk
    // c of row r in slot c ^ swz(r).  K rows are read one per lane (16 rows,
    // the same chunk), V rows four at a time by the transposing reads: each
    // swizzle spreads its 16 lanes over the 16 slots of 256 bytes.
    auto kswz = [](int r) { return CPR == 16 ? r & 15 : CPR == 8 ? (r >> 1) & 7 : (r >> 2) & 3; };
    auto vswz = [](int r) { return CPR == 16 ? 2 * (r & 7) : CPR == 8 ? 2 * ((r >> 1) & 3) : CPR == 4 ? 2 * ((r >> 2) & 1) : 0; };
    uint32_t koff[NL], voff[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        const int cc = 64 * i + lane, row = cc / CPR;
        const int kc = ((cc % CPR) ^ kswz(row)) * 8, vc = ((cc % CPR) ^ vswz(row)) * 8;
        koff[i] = kc < D ? (uint32_t)(((int64_t)row * f.ks + kc) * 2) : 0x80000000u;
        voff[i] = vc < D ? (uint32_t)(((int64_t)row * f.vs + vc) * 2) : 0x80000000u;
    }
    // first key of this wavefront's block of step n (a block outside the valid
    // keys is neither loaded nor computed)
    auto step_key = [&](int n) {
        const int c = n / spc;
        return (c_beg + c) * chunk + 32 * (4 * (n - c * spc) + wave);
    };
    auto live = [&](int n) {
        const int j = step_key(n);
        return n < steps && j <= hi && j + 31 >= lo;
    };
    int page_idx = -1, page_id = 0;
    bool page_ok = false;
    uint16_t* const kt = smem[wave][0];
    uint16_t* const vt = smem[wave][1];
    auto issue = [&](int n, bool k_too, bool v_too) {
        const int j = step_key(n);
        int64_t ko = (int64_t)j * f.ks, vo = (int64_t)j * f.vs;
        int ok = -1;
        if constexpr (PAGED) {
            const int idx = (int)(__umulhi((uint32_t)j, f.page_m) >> f.page_s);
            if (idx != page_idx) {
                page_idx = idx;
                page_id = ((const __attribute__((address_space(4))) int32_t*)(uintptr_t)bt)[idx];
                page_ok = (uint32_t)page_id < (uint32_t)f.npages;
                if (!page_ok) page_id = 0;
            }
            const int64_t jr = j - idx * f.page;
            ko = (int64_t)page_id * f.kb + jr * f.ks;
            vo = (int64_t)page_id * f.vb + jr * f.vs;
            ok = page_ok ? -1 : 0;
        }
        const int rm1 = min(Lk - j, 32) - 1;
        const uint32_t kbytes = __builtin_amdgcn_readfirstlane((int)(((int64_t)rm1 * f.ks + D) * 2) & ok);
        const uint32_t vbytes = __builtin_amdgcn_readfirstlane((int)(((int64_t)rm1 * f.vs + D) * 2) & ok);
        const uint64_t kp = reinterpret_cast<uint64_t>(kbase + ko * 2), vp = reinterpret_cast<uint64_t>(vbase + vo * 2);
        auto load = [&](auto nt) {
            if (k_too) {
#pragma unroll
                for (int i = 0; i < NL; ++i) lds_load16<decltype(nt)::value>(kp, kbytes, kt + 512 * i, koff[i]);
            }
            if (v_too) {
#pragma unroll
                for (int i = 0; i < NL; ++i) lds_load16<decltype(nt)::value>(vp, vbytes, vt + 512 * i, voff[i]);
            }
        };
        if (a.nt)
            load(std::true_type{});
        else
            load(std::false_type{});
    };
    if (live(0)) issue(0, true, true);

    // Q: lane (column l16, group grp) holds head h0 + l16, d = 32 s + 8 grp ..
    op_t qf[DP / 32];
    {
        const char* q = f.q + ((f.cu_q ? u.tok * f.qs : u.b * f.qb) + (int64_t)(u.h0 + l16) * f.qh) * 2;
#pragma unroll
        for (int s = 0; s < DP / 32; ++s) {
            const int d = 32 * s + 8 * grp;
            u32x4_t w = {0, 0, 0, 0};
            if (l16 < u.nr && d < D) w = *reinterpret_cast<const u32x4_t*>(q + d * 2);
            qf[s] = __builtin_bit_cast(op_t, w);
        }
    }
    float slope = f.alibi && l16 < u.nr ? f.alibi[u.b * f.alibi_bstride + u.h0 + l16] : 0.f;
    // (waited for here: a wait inside the loop would drain the K/V loads too)
#pragma unroll
    for (int s = 0; s < DP / 32; ++s) pin(qf[s]);
    pin(slope);
    const float c = a.bias ? kLog2e : f.scale_log2;

    // this wavefront's state of the chunk: column l16's reference and (per
    // lane, its own keys) sum; O^T accumulators (lane: column l16, d = 16 t +
    // 4 grp + 0..3)
    float m = -INFINITY, l = 0.f;
    f32x4_t o[DP / 16];
    auto reset = [&]() {
        m = -INFINITY;
        l = 0.f;
#pragma unroll
        for (int t = 0; t < DP / 16; ++t) o[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    };
    reset();
    // the unit's running sum over chunks: item i of this thread is row
    // (tid + 256 i) / (DP/4), d = 4 ((tid + 256 i) % (DP/4)) ..
    f32x4_t acc[ITEMS];
    float am[ITEMS], al[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        am[i] = -INFINITY;
        al[i] = 0.f;
    }

    // `loaded_v` is called once K is consumed and returns when V has arrived
    auto compute = [&](int j, auto&& loaded_v) {
        // S^T = K Q^T: two 16-key tiles, lane = column, registers = keys
        // j + 16 kk + 4 grp + 0..3
        f32x4_t s[2];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            s[kk] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            const int row = 16 * kk + l16;
#pragma unroll
            for (int d = 0; d < DP / 32; ++d) {
                const op_t ka = *reinterpret_cast<const op_t*>(kt + row * DP + (((4 * d + grp) ^ kswz(row)) << 3));
                s[kk] = O::mfma(ka, qf[d], s[kk]);
            }
        }
        loaded_v();
        if (a.bias) {
            // natural-log units: x = scale*s, soft-cap c tanh(x/c) =
            // c - 2c / (exp(2x/c) + 1), ALiBi
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float x = s[e >> 2][e & 3];
                if (f.softcap > 0.f)
                    x = fmaf(-2.f * f.softcap, __builtin_amdgcn_rcpf(fast_exp2(x * f.softcap_sk) + 1.f), f.softcap);
                else
                    x *= f.scale;
                if (f.alibi) x = fmaf(-slope, fabsf((float)(center - (j + 16 * (e >> 2) + 4 * grp + (e & 3)))), x);
                s[e >> 2][e & 3] = x;
            }
        }
        if (j < lo || j + 31 > hi) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int key = j + 16 * (e >> 2) + 4 * grp + (e & 3);
                s[e >> 2][e & 3] = ((key >= lo) & (key <= hi)) ? s[e >> 2][e & 3] : -INFINITY;
            }
        }
        float mx = s[0][0];
#pragma unroll
        for (int e = 1; e < 8; ++e) mx = fmax_nn(mx, s[e >> 2][e & 3]);
        const float mn = fmax_nn(m, __builtin_ceilf(max_groups(mx) * c));
        const float alpha = pow2_diff(m, mn);
        m = mn;
        const float mu = m == -INFINITY ? 0.f : m;
#pragma unroll
        for (int t = 0; t < DP / 16; ++t) o[t] *= alpha;
        float p[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) p[e] = fast_exp2(fmaf(s[e >> 2][e & 3], c, -mu));
        l = fmaf(l, alpha, ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7])));
        u32x4_t ph, pl;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            uint32_t h, w;
            O::split(p[2 * e], p[2 * e + 1], h, w);
            ph[e] = h;
            pl[e] = w;
        }
        // O^T += V^T P^T: k-slots 0..3 / 4..7 of a group are keys 4 grp + 0..3
        // of the first / second 16
        const int r0 = 4 * grp + (l16 >> 2);
#pragma unroll
        for (int t = 0; t < DP / 16; ++t) {
            const int cb = 2 * t + ((l16 >> 1) & 1);
            const uint16_t* p0 = vt + r0 * DP + ((cb ^ vswz(r0)) << 3) + 4 * (l16 & 1);
            const op_t va = O::load_tr(p0, p0 + 16 * DP);  // (the swizzle of row r0 + 16 is row r0's)
            o[t] = O::mfma(va, __builtin_bit_cast(op_t, ph), o[t]);
            o[t] = O::mfma(va, __builtin_bit_cast(op_t, pl), o[t]);
        }
    };

    const int items = u.nr * (DP / 4);
    for (int n = 0; n < steps; ++n) {
        const bool now = live(n), next = live(n + 1), last = n % spc == spc - 1;
        if (now) {
            wait_vm<NL>();  // (K; V's loads were issued after it)
            compute(step_key(n), [&]() {
                wait_lds();
                if (next) {
                    issue(n + 1, true, false);
                    wait_vm<NL>();
                } else {
                    wait_vm<0>();
                }
            });
        } else if (next) {
            issue(n + 1, true, false);
        }
        wait_lds();
        if (!last) {
            if (next) issue(n + 1, false, true);
            continue;
        }
        // end of a chunk: the wavefronts' sums through their V tiles (consumed;
        // the K tiles may be loading the next chunk), elements 4 c.. of row r at
        // 4 (c ^ (r mod 8))
        l = sum_groups(l);
        float* os = reinterpret_cast<float*>(vt);
        if (l16 < u.nr) {
#pragma unroll
            for (int t = 0; t < DP / 16; ++t)
                *reinterpret_cast<f32x4_t*>(os + l16 * DP + 4 * ((4 * t + grp) ^ (l16 & 7))) = o[t];
            if (grp == 0) {
                m_s[wave][l16] = m;
                l_s[wave][l16] = l;
            }
        }
        // (not __syncthreads: its wait for every load would drain the next chunk's)
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const int it = tid + kDecodeThreads * i;
            if (it < items) {
                const int r = it / (DP / 4), d = 4 * (it % (DP / 4));
                float mc = m_s[0][r];
#pragma unroll
                for (int w = 1; w < 4; ++w) mc = fmax_nn(mc, m_s[w][r]);
                f32x4_t oc = {0.f, 0.f, 0.f, 0.f};
                float lc = 0.f;
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const float e = pow2_diff(m_s[w][r], mc);
                    const f32x4_t x = *reinterpret_cast<const f32x4_t*>(
                        reinterpret_cast<const float*>(smem[w][1]) + r * DP + (d ^ (4 * (r & 7))));
#pragma unroll
                    for (int k = 0; k < 4; ++k) oc[k] = fmaf(x[k], e, oc[k]);
                    lc = fmaf(l_s[w][r], e, lc);
                }
                if (!whole) {  // a partial result, added to the others by the merge kernel
                    const int64_t rows = (int64_t)a.units * a.nr;
                    const int64_t row = (c_beg + n / spc) * rows + (int64_t)unit * a.nr + r;
                    if (d < D) *reinterpret_cast<f32x4_t*>(a.ws_o + row * a.ws_ld + d) = oc;
                    if (d == 0) *reinterpret_cast<float2*>(a.ws_ml + 2 * row) = make_float2(mc, lc);
                    continue;
                }
                // (the merge kernel's arithmetic)
                const float mn = fmax_nn(am[i], mc), e0 = pow2_diff(am[i], mn), e1 = pow2_diff(mc, mn);
#pragma unroll
                for (int k = 0; k < 4; ++k) acc[i][k] = fmaf(oc[k], e1, acc[i][k] * e0);
                al[i] = fmaf(lc, e1, al[i] * e0);
                am[i] = mn;
            }
        }
        reset();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (next) issue(n + 1, false, true);
    }

    if (!whole) return;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const int it = tid + kDecodeThreads * i;
        if (it < items) {
            const int r = it / (DP / 4), d = 4 * (it % (DP / 4));
            if (d < D) store4<IS_BF16>(f, out_row(f, u, r), d, acc[i], al[i]);
            if (d == 0) store_lse(f, u, r, am[i], al[i]);
        }
    }
}

// Sum of a row's chunk results in chunk order, one wavefront per row and 4
// elements per lane (rows whose chunks one workgroup took are already stored).  The references
// and sums of 64 chunks are read at once, one chunk per lane.
template <bool IS_BF16>
__global__ void __launch_bounds__(64) mfa_fwd16x_merge_kernel(DArgs a) {
    const KArgs& f = a.f;
    const int unit = blockIdx.x / a.nr, r = blockIdx.x - unit * a.nr;
    const Unit u = unit_of(a, unit);
    if (u.Lq != 1 || r >= u.nr) return;
    const int n = decode_chunks(u.Lk);
    if (n <= a.group) return;
    const int lane = threadIdx.x, d = 4 * (lane & 31);
    const int64_t rows = (int64_t)a.units * a.nr, row = (int64_t)unit * a.nr + r;
    float m = -INFINITY;
    for (int s = lane; s < n; s += 64) m = fmax_nn(m, a.ws_ml[2 * (s * rows + row)]);
#pragma unroll
    for (int x = 32; x > 0; x >>= 1) m = fmax_nn(m, __shfl_xor(m, x));
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
    float l = 0.f;
    const bool in = d < f.D;
    const float* src = a.ws_o + row * a.ws_ld + (in ? d : 0);
    for (int s0 = 0; s0 < n; s0 += 64) {
        const int sl = s0 + lane;
        float e = 0.f, lw = 0.f;
        if (sl < n) {
            const float2 ml = *reinterpret_cast<const float2*>(a.ws_ml + 2 * (sl * rows + row));
            e = pow2_diff(ml.x, m);
            lw = ml.y;
        }
        const int cnt = min(64, n - s0);
        for (int s1 = 0; s1 < cnt; s1 += 16) {  // (sixteen chunks' loads in flight)
            f32x4_t x[16];
#pragma unroll
            for (int k = 0; k < 16; ++k)
                x[k] = *reinterpret_cast<const f32x4_t*>(src + (s0 + min(s1 + k, cnt - 1)) * rows * a.ws_ld);
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                if (s1 + k < cnt) {
                    const float w = __shfl(e, s1 + k);
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[j] = fmaf(x[k][j], w, acc[j]);
                    l = fmaf(__shfl(lw, s1 + k), w, l);
                }
            }
        }
    }
    if (in && lane < 32) store4<IS_BF16>(f, out_row(f, u, r), d, acc, l);
    if (lane == 0) store_lse(f, u, r, m, l);
}

typedef void (*dfn)(DArgs);
template <int DP, bool IS_BF16>
DecodeKernels kernels_of(bool paged) {
    return DecodeKernels{(void*)(paged ? (dfn)mfa_fwd16x_kernel<DP, IS_BF16, true> : (dfn)mfa_fwd16x_kernel<DP, IS_BF16, false>),
                         (void*)(dfn)mfa_fwd16x_merge_kernel<IS_BF16>, 4 * 2 * 32 * DP * 2 + 2 * 4 * kDecodeRows * 4};
}
template <bool IS_BF16>
DecodeKernels kernels_of(int dp, bool paged) {
    switch (dp) {
        case 32: return kernels_of<32, IS_BF16>(paged);
        case 64: return kernels_of<64, IS_BF16>(paged);
        case 96: return kernels_of<96, IS_BF16>(paged);
        default: return kernels_of<128, IS_BF16>(paged);
    }
}

}  // namespace

DecodeKernels mfa_decode_kernels(int dp, bool bf16, bool paged) {
    return bf16 ? kernels_of<true>(dp, paged) : kernels_of<false>(dp, paged);
}
