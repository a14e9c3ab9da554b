// FlashAttention forward for grids that fwd_kernel's 128-query workgroups leave
// mostly idle: a few query rows over many keys (decoding over a key / value
// cache, short cross-attention) and small batches of short sequences; 16-bit
// inputs, no bias or dropout.
//
// In fwd_kernel one query per head fills 1 of 128 rows, every head of a KV
// group reads its K / V again, and a key loop, a serial chain of tile
// latencies, stays inside one workgroup.  Here
//   * the rows of a workgroup (32) are the (query head of the KV group, query)
//     pairs of one (batch, KV head): K / V are read once for the whole group
//     (with a causal mask, 32 queries of one head);
//   * the keys are split over dec_splits workgroups, and inside one over its 4
//     waves: wave w walks the 64-key tiles t0 + w, t0 + w + 4, ...;
//   * each wave copies its tiles into its own LDS region (direct-to-LDS), so
//     the loop has no barriers: K(t + 4) is copied after the products of S(t),
//     V(t + 4) after those of P(t) V(t), each waited for with a partial vmcnt
//     (the copies of the other matrix stay in flight);
//   * the waves' parts are merged through LDS, the splits' parts (float32,
//     in the caller's workspace) by fwd_combine_kernel.
// Per 64-key tile the arithmetic is fwd_kernel's.  With many keys it is bound
// by the K / V bytes (up to 128 KiB in flight on a CU), with few by the latency
// of the chain of tiles that is left.
// Measured (bf16, D = 128): 16 sequences, 32 query heads on 8 KV heads, 8192
// keys, one query: 224 -> 105 us (2.4 -> 5.1 TB/s of K / V); 1 sequence of them
// 108 -> 22 us; 1 sequence, 32 heads, 32768 keys: 507 -> 119 us.
#pragma once

#include "fa_common.hpp"
#include "fa_params.hpp"

namespace fa {

template <typename T, int D>
struct FwdDecCfg {
    static constexpr int NW = 4;
    static constexpr int NT = 64 * NW;
    static constexpr int BN = 64;                 // keys per tile
    static constexpr int NB = BN / 32;
    static constexpr int KW = D + 8;              // LDS row strides as in FwdCfg
    static constexpr int VW = D + (D == 64 || D == 96 ? 8 : 24);
    static constexpr int KTILE = BN * KW;
    static constexpr int VTILE = BN * VW;
    static constexpr int REGION = KTILE + VTILE;  // elements of a wave's LDS region
    static_assert((D / 32) * 16 * 64 * 4 <= REGION * 2, "a wave's O part fits its region");
};

template <typename T, int D, bool CAUSAL, typename P = FwdParams>
__global__ __launch_bounds__(256, D <= 64 ? 2 : 1) void fwd_decode_kernel(const P p) {
    using C = FwdDecCfg<T, D>;
    static_assert(!Elem<T>::kF32, "16-bit inputs");
    constexpr int BN = C::BN, NB = C::NB, KW = C::KW, VW = C::VW;
    __shared__ __attribute__((aligned(16))) T smem[C::NW * C::REGION];
    __shared__ float stat[C::NW][3][32];  // running max, row sum, raw max of each wave's rows

    const int tid = threadIdx.x;
    const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, hi = lane >> 5;
    // splits of one (batch, KV head, row tile) are consecutive logical ids, so
    // that they run on one XCD's share of the grid
    const int id = xcd_remap((int)blockIdx.x, (int)gridDim.x);
    const int split = id % p.dec_splits;
    const int unit = id / p.dec_splits;  // (batch, KV head, row tile)
    const int rt = unit % p.dec_rt;
    const int bk = unit / p.dec_rt;
    const int hk = bk % p.Hkv, b = bk / p.Hkv;

    const T* __restrict__ kbase = (const T*)p.k + b * p.k_sb + hk * p.k_sh;
    const T* __restrict__ vbase = (const T*)p.v + b * p.v_sb + hk * p.v_sh;
    // ---- this lane's row: (query head g of the group, query i) ----
    const int row = 32 * rt + l32, rg = row / p.dec_sq;
    const bool live = rg < p.group && row - rg * p.dec_sq < p.Sq;
    const int g = live ? rg : 0, i = live ? row - rg * p.dec_sq : 0;
    const int h = hk * p.group + g;
    // key tiles that some row of the unit sees (causal: the unit's rows are
    // consecutive queries of one head)
    int nt = (p.Sk + BN - 1) / BN;
    const int i_first = CAUSAL ? (32 * rt) % p.dec_sq : 0;
    if (CAUSAL) nt = min(nt, min(i_first + 31, p.Sq - 1) / BN + 1);
    const int t0 = (int)((int64_t)nt * split / p.dec_splits), t1 = (int)((int64_t)nt * (split + 1) / p.dec_splits);

    T* Ks = smem + w * C::REGION;
    T* Vs = Ks + C::KTILE;
    DmaTile<T, BN, D, KW, 1> kd;
    kd.init(p.k_ss, lane, 0, ncols<D>(p));
    DmaTile<T, BN, D, VW, 1> vd;
    vd.init(p.v_ss, lane, 0, ncols<D>(p));
    constexpr int NKI = decltype(kd)::NI, NVI = decltype(vd)::NI;
    static_assert(NKI + NVI <= 63, "vmcnt range");
    // tiles past the split's end read nothing (empty range) but are issued, so
    // that the vmcnt counts stay exact
    auto copy_k = [&](int t) FA_INLINE {
        kd.load_untracked(kbase + (int64_t)(t * BN) * p.k_ss, p.k_ss, t < t1 ? p.Sk - t * BN : 0, Ks, lane);
    };
    auto copy_v = [&](int t) FA_INLINE {
        vd.load_untracked(vbase + (int64_t)(t * BN) * p.v_ss, p.v_ss, t < t1 ? p.Sk - t * BN : 0, Vs, lane);
    };

    constexpr int QR = D / 16;
    uint4 qreg[QR];
    {
        const T* qrow = (const T*)p.q + b * p.q_sb + (int64_t)i * p.q_ss + h * p.q_sh;
#pragma unroll
        for (int kk = 0; kk < QR; ++kk)
            qreg[kk] = live && 16 * kk + 8 * hi < ncols<D>(p) ? *reinterpret_cast<const uint4*>(qrow + 16 * kk + 8 * hi)
                                                                 : make_uint4(0u, 0u, 0u, 0u);
    }
    // the Q loads have completed before the copies below are issued: the
    // compiler's own waits for them then never wait for a copy
    wait_vmem();
    asm volatile("" ::: "memory");

    f32x16 o[D / 32];
#pragma unroll
    for (int n = 0; n < D / 32; ++n) o[n] = f32x16{};
    float m_run = -1e30f, l_run = 0.f, m_raw = -INFINITY;
    const float c = p.scale_log2;

    // causal: tiles before n_um are whole for every row of the unit
    const int n_um = CAUSAL ? (i_first + 1) / BN : 0;
    int t = t0 + w;
    copy_k(t);
    copy_v(t);
    for (; t < t1; t += C::NW) {
        // ---- S^T = K Q^T ----
        wait_vmem_below<NVI>();  // K(t); only V(t) may be in flight
        asm volatile("" ::: "memory");
        f32x16 s[NB];
#pragma unroll
        for (int blk = 0; blk < NB; ++blk) {
            s[blk] = f32x16{};
            const T* krow = Ks + (32 * blk + l32) * KW;
#pragma unroll
            for (int kk = 0; kk < QR; ++kk) {
                const s16x8 a = *reinterpret_cast<const s16x8*>(krow + 16 * kk + 8 * hi);
                s[blk] = Elem<T>::mfma(a, __builtin_bit_cast(s16x8, qreg[kk]), s[blk]);
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // K(t) read before it is overwritten
        copy_k(t + C::NW);

        // ---- softmax (as fwd_kernel) ----
        if ((t + 1) * BN > p.Sk || (CAUSAL && t >= n_um)) {
            const int lim = (CAUSAL ? min(p.Sk, i + 1) : p.Sk) - t * BN - 4 * hi;
#pragma unroll
            for (int blk = 0; blk < NB; ++blk)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (32 * blk + 8 * (r >> 2) + (r & 3) >= lim) s[blk][r] = -INFINITY;
        }
        float mx = -INFINITY;
#pragma unroll
        for (int blk = 0; blk < NB; ++blk)
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[blk][r]);
        mx = pair_max(mx);
        m_raw = fmaxf(m_raw, mx);
        const float m_new = fmaxf(m_run, mx * c);
        if (__ballot(m_new > m_run + 8.0f) != 0ull) {
            const float alpha = fast_exp2(m_run - m_new);
            l_run *= alpha;
#pragma unroll
            for (int n = 0; n < D / 32; ++n)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[n][r] *= alpha;
            m_run = m_new;
        }
        float psum = 0.f;
        s16x8 pk[BN / 16];
#pragma unroll
        for (int blk = 0; blk < NB; ++blk)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float pv = fast_exp2(__builtin_fmaf(s[blk][r], c, -m_run));
                psum += pv;
                s[blk][r] = pv;
            }
        l_run += psum;
#pragma unroll
        for (int ks = 0; ks < BN / 16; ++ks) {
            float tmp[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) tmp[e] = s[ks >> 1][8 * (ks & 1) + e];
            pk[ks] = pack8<T>(tmp);
        }

        // ---- O^T += V^T P^T ----
        wait_vmem_below<NKI>();  // V(t); only K(t + 4) may be in flight
        asm volatile("" ::: "memory");
#pragma unroll
        for (int ks = 0; ks < BN / 16; ++ks)
#pragma unroll
            for (int n = 0; n < D / 32; ++n) {
                const T* vp = Vs + (16 * ks + 4 * hi + ((lane & 15) >> 2)) * VW + 32 * n + 16 * ((lane >> 4) & 1) +
                              4 * (lane & 3);
                const s16x8 a = cat4(lds_read_tr16(vp), lds_read_tr16(vp + 8 * VW));
                o[n] = Elem<T>::mfma(a, pk[ks], o[n]);
            }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // V(t) read before it is overwritten
        copy_v(t + C::NW);
    }
    wait_vmem();  // no copy in flight when the region takes the O part
    asm volatile("" ::: "memory");

    // ---- merge the waves' parts (each rescaled to the common maximum) ----
    const float l_w = pair_sum(l_run);
    float* part = reinterpret_cast<float*>(Ks);
#pragma unroll
    for (int n = 0; n < D / 32; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) part[(16 * n + r) * 64 + lane] = o[n][r];
    if (hi == 0) {
        stat[w][0][l32] = m_run;
        stat[w][1][l32] = l_w;
        stat[w][2][l32] = m_raw;
    }
    lds_barrier();
    float mm = stat[0][0][l32];
#pragma unroll
    for (int x = 1; x < C::NW; ++x) mm = fmaxf(mm, stat[x][0][l32]);
    float a[C::NW], l_tot = 0.f;
    m_raw = -INFINITY;
#pragma unroll
    for (int x = 0; x < C::NW; ++x) {
        a[x] = fast_exp2(stat[x][0][l32] - mm);
        l_tot = __builtin_fmaf(stat[x][1][l32], a[x], l_tot);
        m_raw = fmaxf(m_raw, stat[x][2][l32]);
    }
    // wave w merges the 32-column blocks w, w + 4, ...
    f32x16 om;
    const int64_t prow = ((int64_t)unit * p.dec_splits + split) * 32 + l32;  // this row's part
    if (p.dec_splits > 1 && w == 0 && hi == 0) {
        p.dec_stat[prow * 4] = mm;
        p.dec_stat[prow * 4 + 1] = l_tot;
        p.dec_stat[prow * 4 + 2] = m_raw;
    }
    const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    if (p.dec_splits == 1 && w == 0 && hi == 0 && live) {
        const int64_t si = (int64_t)(b * p.H + h) * p.Sq + i;
        p.lse[si] = l_tot > 0.f ? (mm + __log2f(l_tot)) * kLn2 : -INFINITY;
        if (p.mx) p.mx[si] = m_raw * p.scale;
    }
#pragma unroll
    for (int n0 = 0; n0 < D / 32; n0 += C::NW) {
        const int n = n0 + w;
        if (n >= D / 32) break;
#pragma unroll
        for (int r = 0; r < 16; ++r) om[r] = 0.f;
#pragma unroll
        for (int x = 0; x < C::NW; ++x) {
            const float* px = reinterpret_cast<const float*>(smem + x * C::REGION);
#pragma unroll
            for (int r = 0; r < 16; ++r) om[r] = __builtin_fmaf(px[(16 * n + r) * 64 + lane], a[x], om[r]);
        }
        if (p.dec_splits > 1) {
            float* op = p.dec_part + prow * D + 32 * n + 4 * hi;
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4)
                *reinterpret_cast<f32x4*>(op + 8 * q4) = f32x4{om[4 * q4], om[4 * q4 + 1], om[4 * q4 + 2], om[4 * q4 + 3]};
        } else if (live) {
            T* ob = (T*)p.o + b * p.o_sb + (int64_t)i * p.o_ss + h * p.o_sh + 32 * n + 4 * hi;
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                s16x4 v4;
#pragma unroll
                for (int e = 0; e < 4; ++e) v4[e] = Elem<T>::pack1(om[4 * q4 + e] * inv);
                if (32 * n + 8 * q4 < ncols<D>(p)) *reinterpret_cast<s16x4*>(ob + 8 * q4) = v4;
            }
        }
    }
}

// The splits' parts of every row, rescaled to their common maximum and
// normalised: one thread per 4 columns of a row (D / 4 threads share a row).
template <typename T, int D, typename P = FwdParams>
__global__ __launch_bounds__(256) void fwd_combine_kernel(const P p, const int n_rows) {
    constexpr int TPR = D / 4;  // threads per row
    const int gid = (int)blockIdx.x * 256 + (int)threadIdx.x;
    const int r = gid / TPR, col = (gid % TPR) * 4;
    if (r >= n_rows) return;
    // row r = ((b Hkv + hk) group + g) Sq + i, i.e. (b, h, i) in order
    const int bk = r / (p.group * p.Sq), gi = r - bk * (p.group * p.Sq);
    const int rr = gi / p.Sq * p.dec_sq + gi % p.Sq;
    const int64_t base = ((int64_t)(bk * p.dec_rt + (rr >> 5)) * p.dec_splits) * 32 + (rr & 31);
    float mm = -1e30f, m_raw = -INFINITY;
    for (int x = 0; x < p.dec_splits; ++x) {
        mm = fmaxf(mm, p.dec_stat[(base + 32 * x) * 4]);
        m_raw = fmaxf(m_raw, p.dec_stat[(base + 32 * x) * 4 + 2]);
    }
    float l_tot = 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int x = 0; x < p.dec_splits; ++x) {
        const f32x4 st = *reinterpret_cast<const f32x4*>(p.dec_stat + (base + 32 * x) * 4);
        const float a = fast_exp2(st[0] - mm);
        l_tot = __builtin_fmaf(st[1], a, l_tot);
        const f32x4 v = *reinterpret_cast<const f32x4*>(p.dec_part + (base + 32 * x) * D + col);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = __builtin_fmaf(v[e], a, acc[e]);
    }
    const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    const int h = (r / p.Sq) % p.H, b = r / (p.Sq * p.H), i = r % p.Sq;
    if (col == 0) {
        p.lse[r] = l_tot > 0.f ? (mm + __log2f(l_tot)) * kLn2 : -INFINITY;
        if (p.mx) p.mx[r] = m_raw * p.scale;
    }
    s16x4 v4;
#pragma unroll
    for (int e = 0; e < 4; ++e) v4[e] = Elem<T>::pack1(acc[e] * inv);
    if (col < ncols<D>(p)) *reinterpret_cast<s16x4*>((T*)p.o + b * p.o_sb + (int64_t)i * p.o_ss + h * p.o_sh + col) = v4;
}

template <typename T, int D, typename P>
hipError_t launch_fwd_decode_t(const P& p, bool causal, hipStream_t s) {
    const int64_t nb = (int64_t)p.B * p.Hkv * p.dec_rt * p.dec_splits;
    if (causal)
        hipLaunchKernelGGL((fwd_decode_kernel<T, D, true, P>), dim3((unsigned)nb), dim3(256), 0, s, p);
    else
        hipLaunchKernelGGL((fwd_decode_kernel<T, D, false, P>), dim3((unsigned)nb), dim3(256), 0, s, p);
    if (p.dec_splits > 1) {
        const int n_rows = p.B * p.H * p.Sq;
        const int64_t nt = (int64_t)n_rows * (D / 4);
        hipLaunchKernelGGL((fwd_combine_kernel<T, D, P>), dim3((unsigned)((nt + 255) / 256)), dim3(256), 0, s, p, n_rows);
    }
    return hipGetLastError();
}

template <typename T>
hipError_t launch_fwd_decode(const FwdParams& p, int D, bool causal, hipStream_t s) {
    if (p.head_cols > 0) {
        FwdParamsCols pc;
        static_cast<FwdParams&>(pc) = p;
        if (D == 64) return launch_fwd_decode_t<T, 64>(pc, causal, s);
        if (D == 128 && p.head_cols <= 96) return launch_fwd_decode_t<T, 96>(pc, causal, s);
        return D == 128 ? launch_fwd_decode_t<T, 128>(pc, causal, s) : hipErrorInvalidValue;
    }
    switch (D) {
        case 32: return launch_fwd_decode_t<T, 32>(p, causal, s);
        case 64: return launch_fwd_decode_t<T, 64>(p, causal, s);
        case 128: return launch_fwd_decode_t<T, 128>(p, causal, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace fa
