// mfa_bwd32.hip -- fp32 flash-attention backward on the fp32 matrix cores:
// fp32 q, k, v, o and dO in, fp32 dq, dk and dv out, every product and sum in
// fp32 (v_mfma_f32_32x32x2_f32), the fp32 forward's score transform.
//
// The decomposition is that of the 16-bit kernels (mfa_bwd.hip): dQ (and Dsum)
// for a block of query rows, walking the key blocks they see; then dK/dV for a
// block of keys of one (sequence, K/V head), walking every query block of its
// head group that sees them.  No atomics: a fixed order of sums.
//
// What bounds them: the matrix pipe.  One 32 x 32 tile of (query, key) pairs
// is 2 DP MFMAs of 64 cycles in dK/dV (1.5 DP in dQ), against ~300 vector
// instructions and 32 KB of LDS reads at DP = 64.  So the split is made for
// parallel work and short walks, not for operand reuse: a workgroup owns only
// 32 keys (32 query rows), and its four wavefronts take every fourth block of
// the walk, each on its own -- own LDS tiles, no barrier until their sums are
// added at the end.  A tile's loads go straight to LDS and are issued as soon
// as its last reader is done, so that another product's MFMAs cover them.
// Accumulators feed the next product as they are: S and dP come out with
// lane = key (dK/dV) or lane = query (dQ), and register r of P / dS is the
// B operand of an MFMA over the two rows acc_row(r) and acc_row(r) + 4.
// Measured on MI355X (us, against the vector-ALU kernels of 2 x 4 scores per
// thread that these replace): B=2 L=1024 H=8 D=64 causal dK/dV 285 -> 60, dQ
// 158 -> 45; B=1 L=4096 H=16 D=64 dK/dV 1215 and dQ 891 (113 and 116 TFLOP/s of
// products; a large fp32 matrix product reaches 154 on this card).
#include <math.h>
#include <stdint.h>

#include "mfa.h"
#include "mfa_bwd_common.h"
#include "mfa_tile32.h"

namespace {

// Per (sequence, query head) / (sequence, K/V head) rows of fp32 tensors.
struct QView32 {
    const float* q;
    const float* dout;
    const float* o;
    float* dq;
    const float* lse;
    float* dsum;
    int Lq, Lk;
};
__device__ __forceinline__ QView32 q_view32(const BArgs& a, int b, int hq) {
    const KArgs& f = a.f;
    QView32 s;
    int64_t qs = 0, qb = 0;
    if (f.cu_q) {
        const int q0 = f.cu_q[b];
        s.Lq = f.cu_q[b + 1] - q0;
        s.Lk = f.cu_k[b + 1] - f.cu_k[b];
        qs = q0;
        s.lse = f.lse + (int64_t)hq * f.lse_h + q0;
    } else {
        s.Lq = f.Lq;
        s.Lk = f.Lk;
        qb = b;
        s.lse = f.lse + (int64_t)b * f.lse_b + (int64_t)hq * f.lse_h;
    }
    s.q = reinterpret_cast<const float*>(f.q) + (qb * f.qb + qs * f.qs + (int64_t)hq * f.qh);
    s.o = reinterpret_cast<const float*>(f.o) + (qb * f.ob + qs * f.os + (int64_t)hq * f.oh);
    s.dout = reinterpret_cast<const float*>(a.dout) + (qb * a.dob + qs * a.dos + (int64_t)hq * a.doh);
    s.dq = reinterpret_cast<float*>(a.dq) + (qb * a.dqb + qs * a.dqs + (int64_t)hq * a.dqh);
    s.dsum = a.dsum + ((int64_t)b * f.Hq + hq) * f.Lq;
    return s;
}
struct KView32 {
    const float* k;
    const float* v;
    float* dk;
    float* dv;
    int Lk;
};
__device__ __forceinline__ KView32 k_view32(const BArgs& a, int b, int hkv) {
    const KArgs& f = a.f;
    KView32 s;
    int64_t ks = 0, kb = 0;
    if (f.cu_k) {
        ks = f.cu_k[b];
        s.Lk = f.cu_k[b + 1] - f.cu_k[b];
    } else {
        kb = b;
        s.Lk = f.Lk;
    }
    s.k = reinterpret_cast<const float*>(f.k) + (kb * f.kb + ks * f.ks + (int64_t)hkv * f.kh);
    s.v = reinterpret_cast<const float*>(f.v) + (kb * f.vb + ks * f.vs + (int64_t)hkv * f.vh);
    s.dk = reinterpret_cast<float*>(a.dk) + (kb * a.dkb + ks * a.dks + (int64_t)hkv * a.dkh);
    s.dv = reinterpret_cast<float*>(a.dv) + (kb * a.dvb + ks * a.dvs + (int64_t)hkv * a.dvh);
    return s;
}

// Tile of slot t of a grid that takes every unit's tiles from the heaviest to
// the lightest.  Where the whole grid is resident at once, two workgroups on a
// CU (a.fold, set by the host), the slots of the second workgroups run in
// reverse, so a CU pairs a heavy tile with a light one.
__device__ __forceinline__ int fold_slot(const BArgs& a, int t) {
    return a.fold > 0 && t >= a.fold ? a.fold + a.T - 1 - t : t;
}

// P and dS * d score / d (q.k) of one (row, key) pair from s = q.k and dP:
// score = scale*s, soft-cap (precise tanh), ALiBi; P = exp(score - lse).
template <bool BIAS>
__device__ __forceinline__ void pair32(const KArgs& f, float lse2, float dsum, float slope, int dist, bool valid,
                                       float s, float dp, float& p, float& ds) {
    float x = s * f.scale, dx = f.scale;
    if constexpr (BIAS) {
        if (f.softcap > 0.f) {
            const float t = precise_tanh(__fdiv_rn(x, f.softcap));
            x = f.softcap * t;
            dx *= 1.f - t * t;
        }
        if (f.alibi) x = fmaf(-slope, fabsf((float)dist), x);
    }
    p = valid ? fast_exp2(fmaf(x, kLog2e, -lse2)) : 0.f;
    ds = p * (dp - dsum) * dx;
}

// dQ of 32 query rows (lane = row): dQ^T = sum over key blocks of K^T dS'^T
// (dS' = dS * d score / d(q.k)).  Per block: dP^T = V dO^T, S^T = K Q^T, dS',
// dQ^T; V's tile is free after the first product and K's after the last, so
// the next V loads behind S, dS' and dQ and the next K behind dP.
template <int DP, bool BIAS>
__global__ void __launch_bounds__(kBThreads) __attribute__((amdgpu_waves_per_eu(DP <= kB32PairDim ? 2 : 1)))
mfa_bwd32_dq_kernel(BArgs a) {
    typedef Tile<DP> T;
    constexpr int DB = DP / 32;
    __shared__ __attribute__((aligned(16))) float k_s[4][T::FLOATS];
    __shared__ __attribute__((aligned(16))) float v_s[4][T::FLOATS];
    const KArgs& f = a.f;
    const int units = f.B * f.Hq;
    // the last (under a causal mask the heaviest) rows of every unit first
    const int tt = blockIdx.x / units, unit = blockIdx.x - tt * units;
    const int tile = a.T - 1 - fold_slot(a, tt);
    const int b = unit / f.Hq, hq = unit - b * f.Hq;
    const QView32 qv = q_view32(a, b, hq);
    const int Lq = qv.Lq, D = f.D;
    const int q0 = tile * kB32Rows;
    if (q0 >= Lq) return;
    const KView32 kv = k_view32(a, b, hq / (f.Hq / f.Hkv));
    const int Lk = kv.Lk, dq = Lk - Lq;
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nrow = min(kB32Rows, Lq - q0);
    const int row = q0 + l32;
    const bool in = row < Lq;
    const bool kwide = 32 * f.ks * 4 >= ((int64_t)1 << 31), vwide = 32 * f.vs * 4 >= ((int64_t)1 << 31);
    float* kt = k_s[wave];
    float* vt = v_s[wave];

    // key blocks any row of the tile sees (the bounds are monotone in the row)
    const int klo = key_lo(f, q0 + dq), khi = key_hi(f, q0 + nrow - 1 + dq, Lk);
    const int j0 = (klo / 32) * 32;
    const int nblk = khi >= klo ? (khi - j0) / 32 + 1 : 0;
    auto load_k = [&](int it) {
        const int j = j0 + 32 * it;
        T::load(kt, kv.k + (int64_t)j * f.ks, f.ks, min(32, Lk - j), D, lane, kwide);
    };
    auto load_v = [&](int it) {
        const int j = j0 + 32 * it;
        T::load(vt, kv.v + (int64_t)j * f.vs, f.vs, min(32, Lk - j), D, lane, vwide);
    };
    if (wave < nblk) {
        load_v(wave);
        load_k(wave);
    }
    float qf[DP / 2], gf[DP / 2];
    row_operand<DP>(qf, qv.q + (int64_t)row * f.qs, in, D, half);
    row_operand<DP>(gf, qv.dout + (int64_t)row * a.dos, in, D, half);
    const float lse2 = in ? lse2_of(qv.lse[row]) : INFINITY;
    // the row's Dsum = rowsum(dO * O) - dlse, also stored for the dK/dV kernel,
    // which runs after this one
    float dsum = 0.f;
#pragma unroll
    for (int s = 0; s < DP / 2; s += 4) {
        const int d = s + half * (DP / 2);
        float4 w = make_float4(0.f, 0.f, 0.f, 0.f);
        if (in && d < D) w = *reinterpret_cast<const float4*>(qv.o + (int64_t)row * f.os + d);
        dsum = fmaf(w.x, gf[s], dsum);
        dsum = fmaf(w.y, gf[s + 1], dsum);
        dsum = fmaf(w.z, gf[s + 2], dsum);
        dsum = fmaf(w.w, gf[s + 3], dsum);
    }
    dsum = sum_halves(dsum);
    if (in) {
        if (a.dlse) dsum -= a.dlse[(qv.lse - f.lse) + row];  // (same offset as the lse row)
        if (half == 0 && tid < 64) qv.dsum[row] = dsum;
    }
    const int center = row + dq, lo = key_lo(f, center), hi = in ? key_hi(f, center, Lk) : -1;
    const int lo_last = key_lo(f, q0 + nrow - 1 + dq), hi_first = key_hi(f, q0 + dq, Lk);
    const float slope = BIAS && f.alibi ? f.alibi[b * f.alibi_bstride + hq] : 0.f;
    int off[4];
    T::col_offsets(off, l32, half);
    f32x16_t acc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[db][r] = 0.f;

    for (int it = wave; it < nblk; it += 4) {
        const bool more = it + 4 < nblk;
        const int j = j0 + 32 * it;
        f32x16_t s, g;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = g[r] = 0.f;
        wait_vm<T::N>();  // (V's loads were issued before K's)
        T::rows_product(vt, gf, l32, half, g);
        wait_lds();
        wait_vm<0>();
        if (more) load_v(it + 4);
        T::rows_product(kt, qf, l32, half, s);
        auto transform = [&](auto masked_tag) {
            constexpr bool MASKED = decltype(masked_tag)::value;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int key = j + acc_row(r) + 4 * half;
                float p, ds;
                pair32<BIAS>(f, lse2, dsum, slope, center - key, !MASKED || (key >= lo && key <= hi), s[r], g[r], p, ds);
                s[r] = ds;
                // (the soft-cap's temporaries of a few scores at a time, not of all)
                if constexpr (BIAS)
                    if ((r & 3) == 3) __builtin_amdgcn_sched_barrier(0);
            }
        };
        if (nrow == kB32Rows && j >= lo_last && j + 31 <= hi_first)
            transform(std::false_type{});
        else
            transform(std::true_type{});
        T::cols_product(kt, off, s, acc);
        wait_lds();
        if (more) load_k(it + 4);
    }
    T::put(kt, acc, l32, half);
    __syncthreads();
    T::sum4(k_s[0], T::FLOATS, qv.dq + (int64_t)q0 * a.dqs, a.dqs, nrow, D, tid);
}

// dK and dV of 32 keys (lane = key) of one (sequence, K/V head): every query
// block of every query head of the group that sees the keys adds Q^T dS' to
// dK^T and dO^T P to dV^T.  Per block: S = Q K^T, dP = dO V^T, P and dS', dK,
// dV; Q's tile is free after dK and dO's after dV, so the next Q loads behind
// dV and the next dO behind the next S.
template <int DP, bool BIAS>
__global__ void __launch_bounds__(kBThreads) __attribute__((amdgpu_waves_per_eu(DP <= kB32PairDim ? 2 : 1)))
mfa_bwd32_dkdv_kernel(BArgs a) {
    typedef Tile<DP> T;
    constexpr int DB = DP / 32;
    __shared__ __attribute__((aligned(16))) float q_s[4][T::FLOATS];
    __shared__ __attribute__((aligned(16))) float do_s[4][T::FLOATS];
    __shared__ __attribute__((aligned(16))) float stat_s[4][64];  // exp2-domain lse, Dsum of the block's rows
    const KArgs& f = a.f;
    // the first (under a causal mask the heaviest) keys of every unit first
    const int slot = blockIdx.x / a.Ukv, ukv = blockIdx.x - slot * a.Ukv;
    const int b = ukv / f.Hkv, hkv = ukv - b * f.Hkv;
    const KView32 kv = k_view32(a, b, hkv);
    const int Lk = kv.Lk, D = f.D;
    // (a sequence shorter than the longest skips the first slots: the heaviest
    // tiles of all sequences run first)
    const int k0 = (fold_slot(a, slot) - a.T + (Lk + kB32Keys - 1) / kB32Keys) * kB32Keys;
    if (k0 < 0 || k0 >= Lk) return;
    const int nk = min(kB32Keys, Lk - k0), k1 = k0 + nk - 1;
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int key = k0 + l32;
    const int R = f.Hq / f.Hkv;
    const int Lq = f.cu_q ? f.cu_q[b + 1] - f.cu_q[b] : f.Lq;
    const int dq = Lk - Lq;
    const bool qwide = 32 * f.qs * 4 >= ((int64_t)1 << 31), gwide = 32 * a.dos * 4 >= ((int64_t)1 << 31);
    float* qt = q_s[wave];
    float* gt = do_s[wave];
    float* stat = stat_s[wave];

    // query blocks whose rows can see [k0, k1], the same for every head
    int qlo = 0, qhi = Lq - 1;
    if (f.causal) qlo = max(qlo, k0 - dq);
    if (f.wr >= 0) qlo = max(qlo, k0 - f.wr - dq);
    if (f.wl >= 0) qhi = min(qhi, k1 + f.wl - dq);
    const int qb0 = (qlo / 32) * 32;
    const int nqb = qhi >= qb0 ? (qhi - qb0) / 32 + 1 : 0;

    // this wavefront's walk: blocks wave, wave + 4, ... of the R x nqb list,
    // head rr and block qi; `st` is this lane's row statistic of the block
    // loaded last (lse on the lower half, Dsum on the upper)
    float st = 0.f;
    auto load_q = [&](int rr, int qi) {
        const QView32 qv = q_view32(a, b, hkv * R + rr);
        const int q0 = qb0 + 32 * qi, r = q0 + l32;
        st = half ? 0.f : INFINITY;
        if (r < Lq) st = half ? qv.dsum[r] : qv.lse[r];
        T::load(qt, qv.q + (int64_t)q0 * f.qs, f.qs, min(32, Lq - q0), D, lane, qwide);
    };
    auto load_g = [&](int rr, int qi) {
        const QView32 qv = q_view32(a, b, hkv * R + rr);
        const int q0 = qb0 + 32 * qi;
        T::load(gt, qv.dout + (int64_t)q0 * a.dos, a.dos, min(32, Lq - q0), D, lane, gwide);
    };
    auto advance = [&](int& rr, int& qi) {
        qi += 4;
        while (qi >= nqb) {
            qi -= nqb;
            ++rr;
        }
    };
    int rr = 0, qi = wave - 4;
    const bool any = nqb > 0;
    if (any) advance(rr, qi);
    if (any && rr < R) {
        load_q(rr, qi);
        load_g(rr, qi);
    }
    float kf[DP / 2], vf[DP / 2];
    row_operand<DP>(kf, kv.k + (int64_t)key * f.ks, key < Lk, D, half);
    row_operand<DP>(vf, kv.v + (int64_t)key * f.vs, key < Lk, D, half);
    int off[4];
    T::col_offsets(off, l32, half);
    f32x16_t dka[DB], dva[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) dka[db][r] = dva[db][r] = 0.f;

    while (any && rr < R) {
        const int q0 = qb0 + 32 * qi;
        const float slope = BIAS && f.alibi ? f.alibi[b * f.alibi_bstride + hkv * R + rr] : 0.f;
        int nrr = rr, nqi = qi;
        advance(nrr, nqi);
        const bool more = nrr < R;
        f32x16_t s, g;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = g[r] = 0.f;
        wait_vm<T::N>();  // (Q's loads were issued before dO's)
        T::rows_product(qt, kf, l32, half, s);
        wait_vm<0>();
        T::rows_product(gt, vf, l32, half, g);
        stat[lane] = half ? st : lse2_of(st);
        auto transform = [&](auto masked_tag) {
            constexpr bool MASKED = decltype(masked_tag)::value;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float4 l4 = *reinterpret_cast<const float4*>(stat + 8 * i + 4 * half);
                const float4 d4 = *reinterpret_cast<const float4*>(stat + 32 + 8 * i + 4 * half);
                const float lv[4] = {l4.x, l4.y, l4.z, l4.w}, dv[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int r = 4 * i + e, center = q0 + acc_row(r) + 4 * half + dq;
                    bool ok = true;
                    if constexpr (MASKED) ok = (key <= key_hi(f, center, Lk)) & (key >= key_lo(f, center));
                    float p, ds;
                    pair32<BIAS>(f, lv[e], dv[e], slope, center - key, ok, s[r], g[r], p, ds);
                    g[r] = p;
                    s[r] = ds;
                }
                // (the soft-cap's temporaries of a few scores at a time, not of all)
                if constexpr (BIAS) __builtin_amdgcn_sched_barrier(0);
            }
        };
        // (rows past the sequence have lse = +inf: P = 0 in either path)
        if (key_lo(f, q0 + 31 + dq) <= k0 && key_hi(f, q0 + dq, Lk) >= k0 + 31)
            transform(std::false_type{});
        else
            transform(std::true_type{});
        T::cols_product(qt, off, s, dka);
        wait_lds();
        if (more) load_q(nrr, nqi);
        T::cols_product(gt, off, g, dva);
        wait_lds();
        if (more) load_g(nrr, nqi);
        rr = nrr;
        qi = nqi;
    }
    T::put(qt, dka, l32, half);
    T::put(gt, dva, l32, half);
    __syncthreads();
    T::sum4(q_s[0], T::FLOATS, kv.dk + (int64_t)k0 * a.dks, a.dks, nk, D, tid);
    T::sum4(do_s[0], T::FLOATS, kv.dv + (int64_t)k0 * a.dvs, a.dvs, nk, D, tid);
}

template <int DP>
Bwd32Kernels kernels32(bool bias) {
    typedef void (*fn)(BArgs);
    return Bwd32Kernels{
        (void*)(bias ? (fn)mfa_bwd32_dkdv_kernel<DP, true> : (fn)mfa_bwd32_dkdv_kernel<DP, false>),
        (void*)(bias ? (fn)mfa_bwd32_dq_kernel<DP, true> : (fn)mfa_bwd32_dq_kernel<DP, false>)};
}

}  // namespace

Bwd32Kernels mfa_bwd32_kernels(int dp, bool bias) {
    switch (dp) {
        case 32: return kernels32<32>(bias);
        case 64: return kernels32<64>(bias);
        case 96: return kernels32<96>(bias);
        default: return kernels32<128>(bias);
    }
}
