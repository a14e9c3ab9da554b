// Forward, dQ and dK/dV for float32 inputs without a bias on the bf16 matrix
// instructions: every operand is cut into three bf16 pieces (split3) and a
// product is six matrix products of pieces (mfma_split).  A workgroup that
// meets a value out of their range writes a mark (kRedo) in place of its first
// result and nothing else; fwd_kernel, dq_kernel and dkdv_kernel, launched
// after these kernels over the same blocks of rows, compute the marked ones.
//
// fwd_kernel, dq_kernel and dkdv_kernel run float32 on
// v_mfma_f32_32x32x2_f32, whose rate bounds them (fp32 matrix peak is 1/16 of
// bf16); six bf16 products take 0.375 of its time.  Cutting a tile's values
// where each wave reads them would make the vector unit the bound (measured:
// only 6-10% faster), so a tile is cut once per workgroup: each thread loads
// its share of the next tile into registers a tile ahead, cuts it and writes
// the pieces to LDS as rows of [piece 0 | piece 1 | piece 2], which the products
// read like 16-bit tiles (rows, or columns with ds_read_b64_tr_b16).  One LDS
// buffer and two barriers a tile: the workgroups of a CU cover each other's.
// Bound by the matrix products and the splitting of P / dS per tile.
// Error against 64 bits (2-norm of O, dQ, dK, dV at 8 x 1000 x 16 heads of 64):
// full 5.4e-7, 4.7e-7, 4.6e-7, 4.4e-7 (on v_mfma_f32_32x32x2_f32 6.4e-7, 7.6e-7,
// 7.5e-7, 7.3e-7), causal 2.6e-7, 3.6e-7, 3.6e-7, 3.0e-7 (3.3e-7, 4.8e-7, 4.9e-7,
// 4.2e-7).
// Measured (forward / dQ and dK/dV, us; before: on v_mfma_f32_32x32x2_f32; the
// three launches for marked rows, of which there are none here, take 4 to 5 each
// on 1000 workgroups, 1.5 on few):
// 8 x 1000 x 16 heads of 64, full: 288 / 916 -> 203 / 635; causal with dropout,
// heads of 32, 64, 128: 225 / 324, 307 / 595, 457 / 1213 -> 156 / 229, 199 /
// 405, 361 / 993; 4 x 1024 x 16 heads of 128, full: 262 / 982 -> 199 / 686.
// Small grids too: 1 x 512 x 8 heads of 64 39 / 129 -> 35 / 98.
#pragma once

#include "fa_common.hpp"
#include "fa_params.hpp"

namespace fa {

template <int D>
struct F32Cfg {
    static constexpr int NW = 4;
    static constexpr int NT = 64 * NW;
    static constexpr int BM = 32 * NW;  // queries (forward, dQ) or keys (dK/dV) per workgroup
    static constexpr int BN = 32;       // rows of a tile
    // bf16 elements of an LDS row: b128 reads of 8 rows and the transposing
    // reads of 4 rows fall in distinct banks at this stride
    static constexpr int RW = 3 * D + (D == 128 ? 24 : 8);
    static constexpr int TILE = BN * RW;
    static constexpr int OW = 36;  // floats of an output staging row (32 columns)
    static constexpr int SMEM_BYTES = 2 * TILE * 2 > NW * 32 * OW * 4 ? 2 * TILE * 2 : NW * 32 * OW * 4;
    static constexpr int BLOCKS = D == 128 ? 1 : 2;  // workgroups per CU that the registers allow (dQ, dK/dV)
};

// The staging of two [32][D] float32 tiles (rows of `a`, rows of `b`): 8-float
// chunks dealt to the 256 threads, the matrix of an item wave-uniform.
template <int D>
struct F32Stage {
    using C = F32Cfg<D>;
    static constexpr int CPR = D / 8;               // chunks per row
    static constexpr int CH = C::BN * CPR;          // per tile
    static constexpr int PER = 2 * CH / C::NT;      // items per thread
    static_assert(CH % 64 == 0 && 2 * CH % C::NT == 0, "whole waves per matrix");
    uint4 x[PER][2];

    // rows >= nvalid read as zeros
    __device__ FA_INLINE inline void load(const float* a, int64_t sa, const float* b, int64_t sb, int nvalid, int tid) {
        const __amdgpu_buffer_rsrc_t ra = row_buffer<float, D, C::BN>(a, sa, nvalid);
        const __amdgpu_buffer_rsrc_t rb = row_buffer<float, D, C::BN>(b, sb, nvalid);
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const int c = tid + C::NT * u;
            const bool second = __builtin_amdgcn_readfirstlane(c) >= CH;
            const int cc = c - (second ? CH : 0);
            const int off = ((cc / CPR) * (int)(second ? sb : sa) + (cc % CPR) * 8) * 4;
            const __amdgpu_buffer_rsrc_t rs = second ? rb : ra;
            x[u][0] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
            x[u][1] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, off + 16, 0, 0));
        }
    }
    // the pieces into the tiles la, lb
    __device__ FA_INLINE inline void store(bf16* la, bf16* lb, int tid, PieceRange& range) const {
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const int c = tid + C::NT * u;
            const bool second = __builtin_amdgcn_readfirstlane(c) >= CH;
            const int cc = c - (second ? CH : 0);
            bf16* dst = (second ? lb : la) + (cc / CPR) * C::RW + (cc % CPR) * 8;
            const f32x4 p = __builtin_bit_cast(f32x4, x[u][0]), q = __builtin_bit_cast(f32x4, x[u][1]);
            float v[8] = {p[0], p[1], p[2], p[3], q[0], q[1], q[2], q[3]};
            range.add(v);
            const Split3 s = split3(v);
#pragma unroll
            for (int t = 0; t < 3; ++t) *reinterpret_cast<s16x8*>(dst + t * D) = s.p[t];
        }
    }
};

// the pieces of columns 16 kk + 8 hi .. + 7 of one LDS row
template <int D>
__device__ FA_INLINE inline Split3 f32_row_frag(const bf16* row, int kk, int hi) {
    Split3 s;
#pragma unroll
    for (int t = 0; t < 3; ++t) s.p[t] = *reinterpret_cast<const s16x8*>(row + t * D + 16 * kk + 8 * hi);
    return s;
}
// the pieces of column 32 i + l32, rows 16 ks + {4 hi .. + 3, 8 + 4 hi .. + 3}
template <int D>
__device__ FA_INLINE inline Split3 f32_col_frag(const bf16* tile, int ks, int i, int lane, int hi) {
    constexpr int RW = F32Cfg<D>::RW;
    const bf16* p = tile + (16 * ks + 4 * hi + ((lane & 15) >> 2)) * RW + 32 * i + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    Split3 s;
#pragma unroll
    for (int t = 0; t < 3; ++t) s.p[t] = cat4(lds_read_tr16(p + t * D), lds_read_tr16(p + t * D + 8 * RW));
    return s;
}
// a row of D floats in registers: pieces of columns 16 kk + 8 hi .. + 7 (zeros if !ok)
template <int D>
__device__ FA_INLINE inline void f32_row_regs(const float* row, bool ok, int hi, Split3 (&s)[D / 16],
                                                    PieceRange& range) {
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; e += 4) {
            const float4 x = ok ? *reinterpret_cast<const float4*>(row + 16 * kk + 8 * hi + e) : make_float4(0.f, 0.f, 0.f, 0.f);
            v[e] = x.x;
            v[e + 1] = x.y;
            v[e + 2] = x.z;
            v[e + 3] = x.w;
        }
        range.add(v);
        s[kk] = split3(v);
    }
}
// pieces of accumulator values 8 ks .. 8 ks + 7 (P, dS)
__device__ FA_INLINE inline Split3 f32_acc_frag(const f32x16& s, int ks) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = s[8 * ks + e];
    return split3(v);
}
// acc (transposed: lane = row l32, value 4 g + e of block i = column 32 i + 8 g
// + 4 hi + e) times mul to `rows` rows at `out`, 32 columns at a time through
// the wave's staging rows
template <int D>
__device__ FA_INLINE inline void f32_store_rows(float* out, int64_t stride, int rows, const f32x16 (&acc)[D / 32], float mul,
                                                float* stage, int lane, int l32, int hi) {
    constexpr int OW = F32Cfg<D>::OW;
#pragma unroll
    for (int i = 0; i < D / 32; ++i) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = acc[i][4 * g + e] * mul;
            *reinterpret_cast<f32x4*>(stage + l32 * OW + 8 * g + 4 * hi) = v;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int row = 8 * u + (lane >> 3), col = 4 * (lane & 7);
            const f32x4 v = *reinterpret_cast<const f32x4*>(stage + row * OW + col);
            if (row < rows) *reinterpret_cast<f32x4*>(out + (int64_t)row * stride + 32 * i + col) = v;
        }
    }
}

// ---------------------------------------------------------------------------
// Forward: 128 queries of one (batch, head) per workgroup, a query per lane, as
// fwd_kernel (same dropout modes, lazy rescale, LSE).
template <int D, bool CAUSAL, int DROPOUT>
__global__ __launch_bounds__(256, 2) void fwd32_kernel(const FwdParams p) {
    using C = F32Cfg<D>;
    constexpr int BN = C::BN;
    __shared__ __attribute__((aligned(16))) char smem[C::SMEM_BYTES];
    __shared__ __attribute__((aligned(16))) unsigned flags[C::NW];
    bf16* Ks = (bf16*)smem;
    bf16* Vs = Ks + C::TILE;

    const int tid = threadIdx.x;
    const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, hi = lane >> 5;
    const int2 tord = tile_order<64, CAUSAL>(p.n_qtiles);
    const int qt = p.n_qtiles - 1 - tord.y;  // longest causal rows first
    const int h = tord.x % p.H, b = tord.x / p.H;
    const int hk = h / p.group;
    const int q0 = qt * C::BM, qw0 = q0 + 32 * w, qi = qw0 + l32;
    const float* kbase = (const float*)p.k + b * p.k_sb + hk * p.k_sh;
    const float* vbase = (const float*)p.v + b * p.v_sb + hk * p.v_sh;
    int kv_end = p.Sk;
    if (CAUSAL) kv_end = min(kv_end, min(q0 + C::BM, p.Sq));
    const int n_tiles = (kv_end + BN - 1) / BN;
    int n_w = n_tiles;  // tiles this wave uses
    if (CAUSAL) n_w = min(n_tiles, (qw0 + 31) / BN + 1);

    F32Stage<D> st;
    PieceRange range;
    auto load = [&](int j) FA_INLINE {
        const int k0 = j * BN;
        st.load(kbase + (int64_t)k0 * p.k_ss, p.k_ss, vbase + (int64_t)k0 * p.v_ss, p.v_ss, p.Sk - k0, tid);
    };
    if (n_tiles > 0) load(0);
    Split3 qs[D / 16];
    f32_row_regs<D>((const float*)p.q + b * p.q_sb + (int64_t)qi * p.q_ss + h * p.q_sh, qi < p.Sq, hi, qs, range);

    f32x16 o[D / 32];
#pragma unroll
    for (int i = 0; i < D / 32; ++i) o[i] = f32x16{};
    float m_run = -1e30f, l_run = 0.f, m_raw = -INFINITY;
    const float c = p.scale_log2;
    uint64_t row_ctr = 0;
    if (DROPOUT == 1) row_ctr = p.offset + ((uint64_t)(b * p.H + h) * (uint64_t)p.Sq + (uint64_t)qi) * (uint64_t)p.Sk;
    const uint32_t* kbrow = p.kb + (DROPOUT == 2 && qi < p.Sq ? ((int64_t)(b * p.H + h) * p.Sq + qi) * p.kb_w : 0);

    for (int j = 0; j < n_tiles; ++j) {
        const int k0 = j * BN;
        lds_barrier();  // every wave is done with tile j - 1
        st.store(Ks, Vs, tid, range);
        uint32_t kword = 0;
        if (DROPOUT == 2 && qi < p.Sq) kword = kbrow[j];
        if (j + 1 < n_tiles) load(j + 1);
        lds_barrier();
        if (j >= n_w) continue;
        f32x16 s = f32x16{};
        const bf16* krow = Ks + l32 * C::RW;
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) s = mfma_split(f32_row_frag<D>(krow, kk, hi), qs[kk], s);
        if (k0 + BN > p.Sk || (CAUSAL && k0 + BN - 1 > qw0)) {
            const int lim = (CAUSAL ? min(p.Sk, qi + 1) : p.Sk) - k0 - 4 * hi;
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (8 * (r >> 2) + (r & 3) >= lim) s[r] = -INFINITY;
        }
        float mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r]);
        mx = pair_max(mx);
        m_raw = fmaxf(m_raw, mx);
        const float m_new = fmaxf(m_run, mx * c);
        if (__ballot(m_new > m_run + 8.0f) != 0ull) {
            const float alpha = fast_exp2(m_run - m_new);
            l_run *= alpha;
#pragma unroll
            for (int i = 0; i < D / 32; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[i][r] *= alpha;
            m_run = m_new;
        }
        float psum = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float pv = fast_exp2(__builtin_fmaf(s[r], c, -m_run));
            psum += pv;
            s[r] = pv;
            if (DROPOUT) {
                const int kk = 8 * (r >> 2) + 4 * hi + (r & 3);
                const bool keep = DROPOUT == 2 ? ((kword >> kk) & 1u) != 0u
                                               : philox_keep(p.seed, row_ctr + (uint64_t)(k0 + kk), p.keep_thresh);
                if (!keep) s[r] = 0.f;
            }
        }
        l_run += psum;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const Split3 bp = f32_acc_frag(s, ks);
#pragma unroll
            for (int i = 0; i < D / 32; ++i) o[i] = mfma_split(f32_col_frag<D>(Vs, ks, i, lane, hi), bp, o[i]);
        }
    }
    put_odd(flags, range, w, lane);
    lds_barrier();  // every wave is done with the tiles
    if (any_odd<C::NW>(flags)) {
        if (tid == 0) reinterpret_cast<unsigned*>(p.lse)[(int64_t)(b * p.H + h) * p.Sq + q0] = kRedo;
        return;
    }
    const float l_tot = pair_sum(l_run);
    const float inv = l_tot > 0.f ? (DROPOUT ? p.rp : 1.f) / l_tot : 0.f;
    if (hi == 0 && qi < p.Sq) {
        const int64_t si = (int64_t)(b * p.H + h) * p.Sq + qi;
        p.lse[si] = l_tot > 0.f ? (m_run + __log2f(l_tot)) * kLn2 : -INFINITY;
        if (p.mx) p.mx[si] = m_raw * p.scale;
    }
    f32_store_rows<D>((float*)p.o + b * p.o_sb + h * p.o_sh + (int64_t)qw0 * p.o_ss, p.o_ss, p.Sq - qw0, o, inv,
                      (float*)smem + w * 32 * C::OW, lane, l32, hi);
}

// ---------------------------------------------------------------------------
// dQ: 128 queries per workgroup, a query per lane, as dq_kernel (after the
// delta pre-pass).
template <int D, bool CAUSAL, int DROPOUT>
__global__ __launch_bounds__(256, F32Cfg<D>::BLOCKS) void dq32_kernel(const BwdParams p, const int n_qtiles) {
    using C = F32Cfg<D>;
    constexpr int BN = C::BN;
    __shared__ __attribute__((aligned(16))) char smem[C::SMEM_BYTES];
    __shared__ __attribute__((aligned(16))) unsigned flags[C::NW];
    bf16* Ks = (bf16*)smem;
    bf16* Vs = Ks + C::TILE;

    const int tid = threadIdx.x;
    const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, hi = lane >> 5;
    const int2 tord = tile_order<32 * C::BLOCKS, CAUSAL>(n_qtiles);
    const int qt = n_qtiles - 1 - tord.y;
    const int h = tord.x % p.H, b = tord.x / p.H;
    const int hk = h / p.group;
    const int q0 = qt * C::BM, qw0 = q0 + 32 * w, qi = qw0 + l32;
    const float* kbase = (const float*)p.k + b * p.k_sb + hk * p.k_sh;
    const float* vbase = (const float*)p.v + b * p.v_sb + hk * p.v_sh;
    int kv_end = p.Sk;
    if (CAUSAL) kv_end = min(kv_end, min(q0 + C::BM, p.Sq));
    const int n_tiles = (kv_end + BN - 1) / BN;
    int n_w = n_tiles;
    if (CAUSAL) n_w = min(n_tiles, (qw0 + 31) / BN + 1);

    F32Stage<D> st;
    PieceRange range;
    auto load = [&](int j) FA_INLINE {
        const int k0 = j * BN;
        st.load(kbase + (int64_t)k0 * p.k_ss, p.k_ss, vbase + (int64_t)k0 * p.v_ss, p.v_ss, p.Sk - k0, tid);
    };
    if (n_tiles > 0) load(0);
    Split3 qs[D / 16], dos[D / 16];
    f32_row_regs<D>((const float*)p.q + b * p.q_sb + (int64_t)qi * p.q_ss + h * p.q_sh, qi < p.Sq, hi, qs, range);
    f32_row_regs<D>((const float*)p.dout + b * p.do_sb + (int64_t)qi * p.do_ss + h * p.do_sh, qi < p.Sq, hi, dos, range);
    const int64_t wi = ((int64_t)b * p.H + h) * p.ws_stride + qi;  // qi < sq_pad
    const float lse2 = p.lse2[wi], del = p.delta[wi], c = p.scale_log2;
    range.add_delta(del);
    uint64_t row_ctr = 0;
    if (DROPOUT == 1) row_ctr = p.offset + ((uint64_t)(b * p.H + h) * (uint64_t)p.Sq + (uint64_t)qi) * (uint64_t)p.Sk;
    const uint32_t* kbrow = p.kb + (DROPOUT == 2 && qi < p.Sq ? ((int64_t)(b * p.H + h) * p.Sq + qi) * p.kb_w : 0);

    f32x16 dq[D / 32];
#pragma unroll
    for (int i = 0; i < D / 32; ++i) dq[i] = f32x16{};
    for (int j = 0; j < n_tiles; ++j) {
        const int k0 = j * BN;
        lds_barrier();
        st.store(Ks, Vs, tid, range);
        uint32_t kword = 0;
        if (DROPOUT == 2 && qi < p.Sq) kword = kbrow[j];
        if (j + 1 < n_tiles) load(j + 1);
        lds_barrier();
        if (j >= n_w) continue;
        f32x16 s = f32x16{}, dp = f32x16{};
        const bf16* krow = Ks + l32 * C::RW;
        const bf16* vrow = Vs + l32 * C::RW;
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) {
            s = mfma_split(f32_row_frag<D>(krow, kk, hi), qs[kk], s);
            dp = mfma_split(f32_row_frag<D>(vrow, kk, hi), dos[kk], dp);
        }
        const bool need_mask = k0 + BN > p.Sk || (CAUSAL && k0 + BN - 1 > qw0);
        const int lim = (CAUSAL ? min(p.Sk, qi + 1) : p.Sk) - k0 - 4 * hi;
        const uint32_t km = DROPOUT == 2 ? kword >> (4 * hi) : 0u;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float pv = fast_exp2(__builtin_fmaf(s[r], c, -lse2));
            if (need_mask && 8 * (r >> 2) + (r & 3) >= lim) pv = 0.f;
            if (DROPOUT) {
                const int key = k0 + 8 * (r >> 2) + 4 * hi + (r & 3);
                const uint32_t m = DROPOUT == 2 ? bit_mask(km, 8 * (r >> 2) + (r & 3))
                                                : (philox_keep(p.seed, row_ctr + (uint64_t)key, p.keep_thresh) ? ~0u : 0u);
                s[r] = pv * __builtin_fmaf(keep_or_zero(dp[r], m), p.rp, -del);
            } else {
                s[r] = pv * (dp[r] - del);
            }
        }
        // a tile's products summed by themselves, then added: fewer roundings at
        // the size of dQ (error of dQ at 2 x 777 x 8 heads of 64, full: 5.9e-7
        // summed in place, 4.2e-7; on the float32 instruction 5.8e-7)
        const Split3 bs[2] = {f32_acc_frag(s, 0), f32_acc_frag(s, 1)};
#pragma unroll
        for (int i = 0; i < D / 32; ++i) {
            f32x16 t = f32x16{};
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) t = mfma_split(f32_col_frag<D>(Ks, ks, i, lane, hi), bs[ks], t);
#pragma unroll
            for (int r = 0; r < 16; ++r) dq[i][r] += t[r];
        }
    }
    put_odd(flags, range, w, lane);
    lds_barrier();
    float* const out = (float*)p.dq + b * p.dq_sb + h * p.dq_sh;
    if (any_odd<C::NW>(flags)) {
        if (tid == 0) *reinterpret_cast<unsigned*>(out + (int64_t)q0 * p.dq_ss) = kRedo;
        return;
    }
    f32_store_rows<D>(out + (int64_t)qw0 * p.dq_ss, p.dq_ss, p.Sq - qw0, dq, p.scale,
                      (float*)smem + w * 32 * C::OW, lane, l32, hi);
}

// ---------------------------------------------------------------------------
// dK/dV: 128 keys of one (batch, KV head) per workgroup, a key per lane; 32-query
// tiles of Q and dO (with LSE * log2 e and delta) as dkdv_kernel takes them, per
// query head of the group from the last tile down.
template <int D, bool CAUSAL, int DROPOUT>
__global__ __launch_bounds__(256, F32Cfg<D>::BLOCKS) void dkdv32_kernel(const BwdParams p, const int n_ktiles) {
    using C = F32Cfg<D>;
    constexpr int BQ = C::BN;
    __shared__ __attribute__((aligned(16))) char smem[C::SMEM_BYTES];
    __shared__ __attribute__((aligned(16))) float ws[2][BQ];  // LSE * log2 e and delta of the tile
    __shared__ __attribute__((aligned(16))) unsigned flags[C::NW];
    bf16* Qs = (bf16*)smem;
    bf16* Ds = Qs + C::TILE;

    const int tid = threadIdx.x;
    const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, hi = lane >> 5;
    const int2 tord = tile_order<32 * C::BLOCKS, CAUSAL>(n_ktiles);  // key block 0 sees the most queries
    const int hk = tord.x % p.Hkv, b = tord.x / p.Hkv;
    const int k0 = tord.y * C::BM, kw0 = k0 + 32 * w, kj = kw0 + l32;
    const int qt_begin = CAUSAL ? k0 / BQ : 0;
    const int qt_end = (p.Sq + BQ - 1) / BQ;
    const int nq = qt_end > qt_begin ? qt_end - qt_begin : 0;
    const int total = nq * p.group;

    F32Stage<D> st;
    PieceRange range;
    float wx = 0.f;
    auto load = [&](int it) FA_INLINE {
        const int hh = hk * p.group + it / nq, qb0 = (qt_end - 1 - it % nq) * BQ;
        st.load((const float*)p.q + b * p.q_sb + (int64_t)qb0 * p.q_ss + hh * p.q_sh, p.q_ss,
                (const float*)p.dout + b * p.do_sb + (int64_t)qb0 * p.do_ss + hh * p.do_sh, p.do_ss, p.Sq - qb0, tid);
        // qb0 + BQ <= sq_pad; +inf / 0 past Sq
        if (tid < 2 * BQ)
            wx = p.lse2[((int64_t)b * p.H + hh) * p.ws_stride + (tid < BQ ? 0 : p.sq_pad) + qb0 + (tid & (BQ - 1))];
    };
    if (total > 0) load(0);
    Split3 ksp[D / 16], vsp[D / 16];
    f32_row_regs<D>((const float*)p.k + b * p.k_sb + (int64_t)kj * p.k_ss + hk * p.k_sh, kj < p.Sk, hi, ksp, range);
    f32_row_regs<D>((const float*)p.v + b * p.v_sb + (int64_t)kj * p.v_ss + hk * p.v_sh, kj < p.Sk, hi, vsp, range);
    f32x16 dk[D / 32], dv[D / 32];
#pragma unroll
    for (int i = 0; i < D / 32; ++i) {
        dk[i] = f32x16{};
        dv[i] = f32x16{};
    }
    const float c = p.scale_log2;
    for (int it = 0; it < total; ++it) {
        const int hh = hk * p.group + it / nq, qb0 = (qt_end - 1 - it % nq) * BQ;
        lds_barrier();
        st.store(Qs, Ds, tid, range);
        if (tid < 2 * BQ) ws[tid >> 5][tid & (BQ - 1)] = wx;
        if (tid >= BQ && tid < 2 * BQ) range.add_delta(wx);
        // the forward's keep word of query qb0 + l32 for the wave's 32 keys
        uint32_t kword = 0;
        if (DROPOUT == 2 && qb0 + l32 < p.Sq && kw0 < p.Sk)
            kword = p.kb[((int64_t)(b * p.H + hh) * p.Sq + qb0 + l32) * p.kb_w + (kw0 >> 5)];
        if (it + 1 < total) load(it + 1);
        lds_barrier();
        if (CAUSAL && qb0 + BQ <= kw0) continue;  // every query precedes the wave's keys
        f32x16 s = f32x16{}, dp = f32x16{};
        const bf16* qrow = Qs + l32 * C::RW;
        const bf16* drow = Ds + l32 * C::RW;
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) {
            s = mfma_split<true>(f32_row_frag<D>(qrow, kk, hi), ksp[kk], s);
            dp = mfma_split<true>(f32_row_frag<D>(drow, kk, hi), vsp[kk], dp);
        }
        const bool mask = CAUSAL && qb0 < kw0 + 31;
        uint64_t col_ctr = 0;
        if (DROPOUT == 1) col_ctr = p.offset + (uint64_t)(b * p.H + hh) * (uint64_t)p.Sq * (uint64_t)p.Sk + (uint64_t)kj;
        const uint32_t km = DROPOUT == 2 ? transpose32(kword, lane) >> (4 * hi) : 0u;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const f32x4 l4 = *reinterpret_cast<const f32x4*>(&ws[0][8 * g + 4 * hi]);
            const f32x4 d4 = *reinterpret_cast<const f32x4*>(&ws[1][8 * g + 4 * hi]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int r = 4 * g + e, q = qb0 + 8 * g + 4 * hi + e;
                float pv = fast_exp2(__builtin_fmaf(s[r], c, -l4[e]));
                if (mask && q < kj) pv = 0.f;
                float dpv = dp[r], pdv = pv;
                if (DROPOUT) {
                    const bool keep = DROPOUT == 2 ? ((km >> (8 * g + e)) & 1u) != 0u
                                                   : philox_keep(p.seed, col_ctr + (uint64_t)q * (uint64_t)p.Sk, p.keep_thresh);
                    dpv = keep ? dpv : 0.f;
                    pdv = keep ? pv : 0.f;
                }
                s[r] = pdv;
                dp[r] = DROPOUT ? pv * __builtin_fmaf(dpv, p.rp, -d4[e]) : pv * (dpv - d4[e]);
            }
        }
        // (each tile's products summed by themselves, as dq32_kernel does: 1-5% of
        // the time; error of dK at 8 x 1000 x 16 heads of 64, causal: 4.2e-7 in
        // place, 3.6e-7)
        auto add = [&](f32x16 (&acc)[D / 32], const bf16* tile, const f32x16& x) FA_INLINE {
            const Split3 bx[2] = {f32_acc_frag(x, 0), f32_acc_frag(x, 1)};
#pragma unroll
            for (int i = 0; i < D / 32; ++i) {
                f32x16 t = f32x16{};
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) t = mfma_split(f32_col_frag<D>(tile, ks, i, lane, hi), bx[ks], t);
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][r] += t[r];
            }
        };
        add(dv, Ds, s);
        add(dk, Qs, dp);
    }
    put_odd(flags, range, w, lane);
    lds_barrier();
    float* const out = (float*)p.dk + b * p.dk_sb + hk * p.dk_sh;
    if (any_odd<C::NW>(flags)) {
        if (tid == 0) *reinterpret_cast<unsigned*>(out + (int64_t)k0 * p.dk_ss) = kRedo;
        return;
    }
    float* stage = (float*)smem + w * 32 * C::OW;
    f32_store_rows<D>(out + (int64_t)kw0 * p.dk_ss, p.dk_ss, p.Sk - kw0, dk, p.scale,
                      stage, lane, l32, hi);
    f32_store_rows<D>((float*)p.dv + b * p.dv_sb + hk * p.dv_sh + (int64_t)kw0 * p.dv_ss, p.dv_ss, p.Sk - kw0, dv,
                      DROPOUT ? p.rp : 1.f, stage, lane, l32, hi);
}

}  // namespace fa
