// The small-M product of fragment-packed or row-major operands: one workgroup's
// work, shared by the panel kernels of kr_gemm.hip and the stepped layers'
// products that carry a row copy (kr_step.hip).
#pragma once
#include <type_traits>

#include "kr_gemm.h"
#include "kr_gemm_epilogue.h"
#include "kr_math.h"
#include "kr_wave.h"

namespace {

constexpr int kKS = KR_GEMM_KSPLIT;

// ---------------------------------------------------------------------------
// Panel kernel (small M)
// ---------------------------------------------------------------------------

// One workgroup per (16*TM) x (16*NS) output tile of one job, one wave per
// 256-wide K slice (S = K/256 waves). A wave loads its slice of the TM A
// fragments once, then streams NS weight panels of 16 columns (double
// buffered), running one 8-deep MFMA chain per (row block, panel). The slice
// partials meet in LDS; the TM*NS result tiles are then shared out over the
// waves, each adding the S partials of a tile in slice order and applying the
// job's epilogue. Several jobs with the same M and K (e.g. the K, V, R
// projections) share one launch.
//
// Time on MI355X is set by the L2 requests a CU has in flight (about 64 lines
// at ~470 cycles each), so the tile shape is chosen on the host to minimise
// the operand bytes the busiest CU reads: a larger NS re-reads A less often.
//
// FRAG: A and W^T are fragment-packed (kr_frag_index), so every operand load
// is one contiguous 1 KB read per wave; otherwise they are row-major and each
// load gathers 16 rows x 64 bytes (about 3x slower).
//
// The MFMA is issued as W^T x A^T, i.e. the weight fragment in the A-operand
// slot: the result lane then holds 4 consecutive output columns of one row,
// so the epilogue reads and writes 8-byte (fp16) or 16-byte (fp32) vectors.
// Every output element is still the same k-ordered chain of products.
//
// Workgroup -> tile: when a job has a multiple of 8 column groups, the
// workgroups of one column group (which share its weight panels) all land on
// the same XCD (workgroups are dealt to the 8 XCDs round robin), so each
// weight byte is fetched into one L2.
//
// QA (w8a8, a_q16): A arrives as fp16 in the fp16 fragment layout and is
// quantised here, one scale per row: each wave takes max |x| over its slice
// of its rows, the waves meet in LDS for the row maximum, and every wave
// rounds its own slice to int8 (kr_q8_pack4) in registers. For finite
// activations the bits are those of kr_quantize_rows followed by the int8
// product, without the separate quantisation launch; the cost is twice the A
// bytes. (The maximum compares fp16 bit patterns, so a NaN outranks every
// finite value here, where kr_quantize_rows' fmaxf skips it.)
constexpr int kEpiPrefetch = 4;   // epilogue tiles per wave with prefetched res/gate

typedef unsigned short kr_u16x2 __attribute__((ext_vector_type(2)));

// Jobs: kr_gemm_multi, or a struct with its fields for one job. COPY (one job
// only): a row copy rides along (copy is not read otherwise). Its code costs a
// panel launch four registers and ~0.1 us (and the 2 x 2 tile a wave per SIMD:
// the channel-mix R/K product at 176 rows 7.0 -> 8.2 us on MI355X), so the
// launches with one are kernels of their own (kr_step.hip). mj is taken by
// value: by reference the kernel arguments are loaded and selected in another
// order (12 layers of 7 rows, C = 768, MI355X: 363 against 355 us; w8a8,
// C = 512, 192 rows 389 / 384).
template <int TM, int NS, bool FRAG, bool I8, bool QA, bool COPY, class Jobs>
__device__ __forceinline__ void panel_product(Jobs mj, kr_row_copy copy) {
    static_assert(!QA || (I8 && FRAG), "on-load quantisation needs the int8 fragment path");
    constexpr int TT = TM * NS;
    // 1 KB operand blocks per wave slice: 8 x (16x32 fp16) or 4 x (16x64 int8);
    // either way a wave covers 256 k. int8 operands move as 16-bit pairs.
    constexpr int QPS = I8 ? 4 : 8;
    typedef typename std::conditional<I8, kr_int4, kr_float4>::type Acc;
    extern __shared__ __attribute__((aligned(16))) float part_lds[];   // [S][TT][256]
    const int lane = threadIdx.x & 63, s = threadIdx.x >> 6;
    // decode-step timing only (stamps non-null): this wave's start and end
    const unsigned long long t_start = mj.stamps ? (unsigned long long)wall_clock64() : 0ull;
    auto stamp_end = [&]() {
        if (mj.stamps && lane == 0) {
            typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
            *reinterpret_cast<u64x2*>(mj.stamps + 2 * (KR_STAMP_WAVES * blockIdx.x + s)) =
                u64x2{t_start, (unsigned long long)wall_clock64()};
        }
    };
    // Job of this workgroup; fields are copied with constant indices so every
    // kernel-argument load is issued up front (no dependent scalar loads).
    const int bid = blockIdx.x;
    kr_gemm_args g;
    int ep, w;
    if constexpr (COPY) {
        w = bid;
        g = mj.job[0];
        ep = mj.ep[0];
    } else {
        const int j = bid < mj.tiles[0] ? 0 : (bid < mj.tiles[0] + mj.tiles[1] ? 1 : 2);
        w = bid - (j > 0 ? mj.tiles[0] : 0) - (j > 1 ? mj.tiles[1] : 0);
        if (j == 0) { g = mj.job[0]; ep = mj.ep[0]; }
        else if (j == 1) { g = mj.job[1]; ep = mj.ep[1]; }
        else { g = mj.job[2]; ep = mj.ep[2]; }
    }
    const int S = g.K / kKS;
    const int mt = (g.M + 16 * TM - 1) / (16 * TM);
    const int ng = (g.N + 16 * NS - 1) / (16 * NS);
    int m_t, n_g;
    if ((ng & 7) == 0) {
        const int k = w >> 3;
        n_g = (k / mt) * 8 + (w & 7);
        m_t = k % mt;
    } else {
        m_t = w / ng;
        n_g = w % ng;
    }
    const int m0 = m_t * 16 * TM, n0 = n_g * 16 * NS;
    const int last_mb = (g.M - 1) >> 4, last_nb = (g.N - 1) >> 4;
    const long long lda16 = I8 ? g.lda >> 1 : g.lda, ldw16 = I8 ? g.ldw >> 1 : g.ldw;

    // ---- operand loads: A once, W panels double buffered (int8, and fp16
    // with three panels of one row block: all NS panels loaded up front)
    constexpr int NB = (I8 || NS == 3) ? NS : 2;
    kr_half8 a[TM][QPS];
    kr_half8 b[NB][QPS];
    // QA: int8 block q of the slice holds, in lane (r, j) = (l % 16, l / 16),
    // the 16 halves k = 64q + 16j .. +15 of row r: fp16 block 2q + j/2 of the
    // slice, lanes r + 32(j % 2) and r + 32(j % 2) + 16.
    kr_half8 af[QA ? TM : 1][QA ? QPS : 1][2];
    const int kb = (I8 ? g.K >> 1 : g.K) >> 5;   // 1 KB blocks per row
    auto load_w = [&](int t, kr_half8 (&dst)[QPS]) {
        // panels beyond N re-read the last one; their outputs are never stored
        if constexpr (FRAG) {
            const int nb = min((n0 >> 4) + t, last_nb);
            const kr_half* bp = g.Wf + ((size_t)nb * kb + QPS * s) * 512 + lane * 8;
            #pragma unroll
            for (int q = 0; q < QPS; q++) dst[q] = *reinterpret_cast<const kr_half8*>(bp + 512 * q);
        } else {
            const int r = min(n0 + 16 * t + (lane & 15), g.N - 1);
            const kr_half* bp = g.Wt + (size_t)r * ldw16 + s * QPS * 32 + (lane >> 4) * 8;
            #pragma unroll
            for (int q = 0; q < QPS; q++) dst[q] = *reinterpret_cast<const kr_half8*>(bp + 32 * q);
        }
    };
    #pragma unroll
    for (int i = 0; i < TM; i++) {
        if constexpr (QA) {
            const int mb = min((m0 >> 4) + i, last_mb), j16 = lane >> 4;
            const kr_half* ap = g.A + ((size_t)mb * (g.K >> 5) + 8 * s + (j16 >> 1)) * 512 +
                                ((lane & 15) + 32 * (j16 & 1)) * 8;
            #pragma unroll
            for (int q = 0; q < QPS; q++) {
                af[i][q][0] = *reinterpret_cast<const kr_half8*>(ap + 1024 * q);
                af[i][q][1] = *reinterpret_cast<const kr_half8*>(ap + 1024 * q + 128);
            }
        } else if constexpr (FRAG) {
            const int mb = min((m0 >> 4) + i, last_mb);
            const kr_half* ap = g.A + ((size_t)mb * kb + QPS * s) * 512 + lane * 8;
            #pragma unroll
            for (int q = 0; q < QPS; q++) a[i][q] = *reinterpret_cast<const kr_half8*>(ap + 512 * q);
        } else {
            const int r = min(m0 + 16 * i + (lane & 15), g.M - 1);
            const kr_half* ap = g.A + (size_t)r * lda16 + s * QPS * 32 + (lane >> 4) * 8;
            #pragma unroll
            for (int q = 0; q < QPS; q++) a[i][q] = *reinterpret_cast<const kr_half8*>(ap + 32 * q);
        }
    }
    #pragma unroll
    for (int t = 0; t < (NB < NS ? NB : NS); t++) load_w(t, b[t]);

    // ---- epilogue operands of this wave's tiles (t = s, s + S, ...), fetched
    // behind the operand loads. The vector path needs 4-column groups that
    // never straddle N and aligned pointers.
    const bool has_res = ep == KR_EP_RESID || ep == KR_EP_GATED;
    const uintptr_t ovec = ep == KR_EP_F32 ? 15 : 7;
    const bool vec = g.out_frag ||
                     ((g.N & 3) == 0 && (g.ldo & 3) == 0 && ((uintptr_t)g.out & ovec) == 0 &&
                      (!has_res || ((uintptr_t)g.res & 7) == 0) &&
                      (ep != KR_EP_GATED || ((uintptr_t)g.gate & 7) == 0));
    const int my_tiles = s < TT ? (TT - 1 - s) / S + 1 : 0;
    const bool prefetch = has_res && vec && my_tiles <= kEpiPrefetch;
    kr_half4 res_v[kEpiPrefetch], gate_v[kEpiPrefetch];
    auto tile_mn = [&](int t, int& m, int& nb) {
        m = m0 + 16 * (t / NS) + (lane & 15);
        nb = n0 + 16 * (t % NS) + 4 * (lane >> 4);
    };
    if (prefetch) {
        const kr_half* gp = ep == KR_EP_GATED ? g.gate : g.res;
        #pragma unroll
        for (int e = 0; e < kEpiPrefetch; e++) {
            if (e < my_tiles) {
                int m, nb;
                tile_mn(s + e * S, m, nb);
                const size_t o = (size_t)min(m, g.M - 1) * (size_t)g.ldo + (size_t)min(nb, g.N - 4);
                res_v[e] = *reinterpret_cast<const kr_half4*>(g.res + o);
                gate_v[e] = *reinterpret_cast<const kr_half4*>(gp + o);
            }
        }
    }
    // ---- row copy: this thread's first unit fetched here, stored at the end
    // (blockDim would be fetched from memory behind the operands, and waited for)
    const int cp0 = bid * 64 * S + (int)threadIdx.x;
    uint2 cp_v;
    if (COPY && cp0 < copy.n) cp_v = copy.src[cp0];
    auto copy_rows = [&]() {
        if (!COPY || cp0 >= copy.n) return;
        copy.dst[cp0] = cp_v;
        const int all = mj.tiles[0] * 64 * S;
        for (int u = cp0 + all; u < copy.n; u += all) copy.dst[u] = copy.src[u];
    };
    __builtin_amdgcn_sched_barrier(0);     // loads in flight before the MFMAs

    // ---- QA: row maxima over all slices, then this slice rounded to int8
    float amax_r[TM];                      // QA: row maximum, then row scale
    if constexpr (QA) {
        float* qmax = part_lds + (size_t)S * TT * 256;     // [S][TM][16]
        #pragma unroll
        for (int i = 0; i < TM; i++) {
            // |x| as fp16 bit patterns: unsigned order is value order (finite x)
            kr_u16x2 m2 = {0, 0};
            #pragma unroll
            for (int q = 0; q < QPS; q++)
                #pragma unroll
                for (int h = 0; h < 2; h++) {
                    const kr_int4 w4 = __builtin_bit_cast(kr_int4, af[i][q][h]);
                    #pragma unroll
                    for (int d = 0; d < 4; d++)
                        m2 = __builtin_elementwise_max(
                            m2, __builtin_bit_cast(kr_u16x2, (unsigned)w4[d] & 0x7fff7fffu));
                }
            unsigned mm = m2[0] > m2[1] ? m2[0] : m2[1];
            mm = max(mm, kr_xor<16>(mm));
            mm = max(mm, kr_xor<32>(mm));
            amax_r[i] = (float)__builtin_bit_cast(kr_half, (unsigned short)mm);
            if (S > 1 && lane < 16) qmax[(s * TM + i) * 16 + lane] = amax_r[i];
        }
        if (S > 1) {
            __syncthreads();
            #pragma unroll
            for (int i = 0; i < TM; i++) {
                float am = qmax[i * 16 + (lane & 15)];
                for (int q = 1; q < S; q++) am = fmaxf(am, qmax[(q * TM + i) * 16 + (lane & 15)]);
                amax_r[i] = am;
            }
        }
        #pragma unroll
        for (int i = 0; i < TM; i++) {
            const float inv = kr_q8_inv(amax_r[i]);
            const float sc = kr_q8_scale(amax_r[i]);
            #pragma unroll
            for (int q = 0; q < QPS; q++) {
                kr_int4 w4;
                #pragma unroll
                for (int d = 0; d < 4; d++) {
                    const kr_half8& h = af[i][q][d >> 1];
                    const int e = 4 * (d & 1);
                    w4[d] = (int)kr_q8_pack4((float)h[e], (float)h[e + 1], (float)h[e + 2],
                                             (float)h[e + 3], inv);
                }
                a[i][q] = __builtin_bit_cast(kr_half8, w4);
            }
            amax_r[i] = sc;                // from here on: the row's scale
        }
    }

    // ---- MFMA chains, one per (row block, panel)
    Acc p[TM][NS];
    #pragma unroll
    for (int t = 0; t < NS; t++) {
        #pragma unroll
        for (int i = 0; i < TM; i++) {
            p[i][t] = Acc{0, 0, 0, 0};
            #pragma unroll
            for (int q = 0; q < QPS; q++) {
                if constexpr (I8)
                    p[i][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(as_i4(b[t % NB][q]),
                                                                   as_i4(a[i][q]), p[i][t], 0, 0, 0);
                else
                    p[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[t % NB][q], a[i][q], p[i][t],
                                                                    0, 0, 0);
            }
        }
        if (t + NB < NS) load_w(t + NB, b[t % NB]);
    }
    // int8: exact int32 sums dequantised once per output
    auto dequant = [&](int t, kr_int4 acc) -> kr_float4 {
        int m, nb;
        tile_mn(t, m, nb);
        float sa;
        if constexpr (QA) {
            // the lane's row of row block t / NS is the one amax_r holds
            sa = amax_r[0];
            #pragma unroll
            for (int i = 1; i < TM; i++)
                if (t / NS == i) sa = amax_r[i];
        } else {
            sa = g.sa[min(m, g.M - 1)];
        }
        kr_float4 y;
        #pragma unroll
        for (int r = 0; r < 4; r++) y[r] = __fmul_rn(__fmul_rn((float)acc[r], sa), g.sw[min(nb + r, g.N - 1)]);
        return y;
    };

    // ---- slice partials in LDS, then each tile summed in slice order
    auto epilogue = [&](int t, int e, kr_float4 acc) {
        int m, nb;
        tile_mn(t, m, nb);
        if (m >= g.M || nb >= g.N) return;
        const size_t o = (size_t)m * (size_t)g.ldo + (size_t)nb;
        if (vec) {
            if (ep == KR_EP_F32) {
                *reinterpret_cast<kr_float4*>(reinterpret_cast<float*>(g.out) + o) = acc;
                return;
            }
            kr_half4 rv = kr_half4{0, 0, 0, 0}, gv = kr_half4{0, 0, 0, 0};
            if (has_res) {
                if (prefetch) {
                    #pragma unroll
                    for (int x = 0; x < kEpiPrefetch; x++)
                        if (x == e) { rv = res_v[x]; gv = gate_v[x]; }
                } else {
                    rv = *reinterpret_cast<const kr_half4*>(g.res + o);
                    if (ep == KR_EP_GATED) gv = *reinterpret_cast<const kr_half4*>(g.gate + o);
                }
            }
            kr_half4 h;
            #pragma unroll
            for (int r = 0; r < 4; r++) {
                const float x = (float)kr_f16(acc[r]);
                float y;
                if (ep == KR_EP_F16) y = x;
                else if (ep == KR_EP_SIGMOID) y = kr_sigmoid_t<I8>(x);
                else if (ep == KR_EP_RELUSQ) { const float rr = x > 0.0f ? x : 0.0f; y = rr * rr; }
                else if (ep == KR_EP_RESID) y = (float)rv[r] + x;
                else y = (float)rv[r] + (float)kr_f16((float)gv[r] * x);
                h[r] = kr_f16(y);
            }
            kr_half* dst = reinterpret_cast<kr_half*>(g.out) +
                           (g.out_frag ? kr_frag_index(m, nb, g.N) : o);
            *reinterpret_cast<kr_half4*>(dst) = h;
        } else {
            #pragma unroll
            for (int r = 0; r < 4; r++)
                if (nb + r < g.N) {
                    switch (ep) {
                        case KR_EP_F32: store_one<KR_EP_F32, I8>(g, m, nb + r, acc[r]); break;
                        case KR_EP_F16: store_one<KR_EP_F16, I8>(g, m, nb + r, acc[r]); break;
                        case KR_EP_SIGMOID: store_one<KR_EP_SIGMOID, I8>(g, m, nb + r, acc[r]); break;
                        case KR_EP_RELUSQ: store_one<KR_EP_RELUSQ, I8>(g, m, nb + r, acc[r]); break;
                        case KR_EP_RESID: store_one<KR_EP_RESID, I8>(g, m, nb + r, acc[r]); break;
                        default: store_one<KR_EP_GATED, I8>(g, m, nb + r, acc[r]); break;
                    }
                }
        }
    };
    if (S == 1) {
        #pragma unroll
        for (int t = 0; t < TT; t++) {
            if constexpr (I8) epilogue(t, t, dequant(t, p[t / NS][t % NS]));
            else epilogue(t, t, p[t / NS][t % NS]);
        }
        copy_rows();
        stamp_end();
        return;
    }
    #pragma unroll
    for (int t = 0; t < TT; t++)
        *reinterpret_cast<Acc*>(part_lds + ((size_t)s * TT + t) * 256 + lane * 4) = p[t / NS][t % NS];
    __syncthreads();
    for (int e = 0; e < my_tiles; e++) {
        const int t = s + e * S;
        Acc acc = *reinterpret_cast<const Acc*>(part_lds + (size_t)t * 256 + lane * 4);
        for (int q = 1; q < S; q++)
            acc = acc + *reinterpret_cast<const Acc*>(part_lds + ((size_t)q * TT + t) * 256 + lane * 4);
        if constexpr (I8) epilogue(t, e, dequant(t, acc));
        else epilogue(t, e, acc);
    }
    copy_rows();
    stamp_end();
}

}  // namespace
