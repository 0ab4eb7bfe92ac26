// Stepped (T = 1) layer products with the LayerNorm-mix that feeds them in
// the same launch, for few streams (kr_step_fuse_ok). The decode step at these
// sizes is a chain of dependent launches, each a memory round trip and a
// dispatch, and these two kernels take two of a layer's six away.
//
// A workgroup takes 16 rows (streams) x a run of output columns. Its waves
// first request their rows and coefficients, then their weight fragments, and
// run LN and the mixes of the workgroup's rows while the weights arrive; the
// mixes (w8a8: quantised per row) meet in LDS, row-major with a 16-byte pad
// (a fragment read then hits 64 distinct banks), and the MFMA chains read
// them from there. Every column group repeats the LN of its rows, about
// 0.13 us of issue per row, which is what bounds the range of M.
//
// The carried row (state) is read by every column group, so the new one goes
// to pend, which the following product copies over it (gemm_panel_copy_kernel).
//
// Same operations in the same order as ln_mix_kernel, kvr_wkv_kernel and
// gemm_panel_kernel: same bits.
//
// Bound: the launch chain (about 4.5 us per launch, 50 launches per step).
// Measured on MI355X, decode step, us, C = 768, six launches per layer / four:
// fp16 B = 1 325 / 276, 8 352 / 315, 16 342 / 332, 40 360 / 328, 80 387 / 353,
// 128 422 / 393, 160 438 / 451, 200 475 / 568; w8a8 B = 1 359 / 290,
// 16 368 / 361, 40 387 / 364, 128 442 / 405, 144 440 / 455, 200 495 / 595.
#include <hip/hip_ext.h>

#include <algorithm>
#include <type_traits>

#include "kr_gemm_epilogue.h"
#include "kr_panel.h"
#include "kr_rowops.h"
#include "kr_step.h"
#include "kr_wkv.h"

namespace {

// 16 rows x C mixes in LDS: bytes from one row to the next.
template <int G, bool Q8>
constexpr int kMixPitch = 256 * G * (Q8 ? 1 : 2) + 16;

template <int G, int NM, int RPW>
struct LnHeld {
    CoefH<G> w, bias, tm[NM], cur[RPW], prev[RPW];
};

// Rows wave, wave + NW, ... of the workgroup's 16 (clamped to the last one)
// and the coefficients, requested.
template <int G, int NM, int RPW, int NW>
__device__ __forceinline__ void ln_request(const kr_step_ln& a, const kr_half* const (&tm)[NM], int m0,
                                           int M, int wave, int lane, LnHeld<G, NM, RPW>& h) {
    constexpr int C = 256 * G;
    #pragma unroll
    for (int u = 0; u < RPW; u++) {
        const size_t m = (size_t)min(m0 + wave + NW * u, M - 1);
        load_coef<G>(a.x + m * C, lane, h.cur[u]);
        load_coef<G>(a.state + m * C, lane, h.prev[u]);
    }
    load_coef<G>(a.ln_w, lane, h.w);
    load_coef<G>(a.ln_b, lane, h.bias);
    #pragma unroll
    for (int m = 0; m < NM; m++) load_coef<G>(tm[m], lane, h.tm[m]);
}

template <int G>
__device__ __forceinline__ void keep_packed(CoefH<G>& c) {
    #pragma unroll
    for (int i = 0; i < G; i++) {
        unsigned long long v = __builtin_bit_cast(unsigned long long, c.v[i]);
        asm volatile("" : "+v"(v));
        c.v[i] = __builtin_bit_cast(kr_half4, v);
    }
}

// LN and mixes of those rows into LDS (mix m of row r at (16 m + r) pitch;
// Q8: its scale at sc[16 m + r]); pend rows written by one column group.
template <int G, int NM, int RPW, int NW, bool Q8>
__device__ __forceinline__ void ln_mix_lds(LnHeld<G, NM, RPW>& h, kr_half* pend, int m0, int M,
                                           int wave, int lane, char* mix, float* sc) {
    constexpr int C = 256 * G;
    #pragma unroll
    for (int u = 0; u < RPW; u++) {
        const int r = wave + NW * u;
        if (r >= 16 || m0 + r >= M) break;         // wave-uniform
        RowF<G> cur, prev;
        to_float<G>(h.cur[u], cur);
        to_float<G>(h.prev[u], prev);
        layer_norm_row<G>(cur, h.w, h.bias);
        #pragma unroll
        for (int m = 0; m < NM; m++) {
            char* row = mix + (16 * m + r) * kMixPitch<G, Q8>;
            if constexpr (Q8)
                store_mix_q8<G>(reinterpret_cast<int8_t*>(row), sc + 16 * m + r, 0, false, h.tm[m], lane,
                                cur, prev);
            else
                store_mix<G>(reinterpret_cast<kr_half*>(row), 0, false, h.tm[m], lane, cur, prev);
        }
        if (pend) store_row<G>(pend + (size_t)(m0 + r) * C, lane, cur);
        // one row's registers at a time: without this the coefficients' fp32
        // copies live across the rows (spills beside the held weights)
        keep_packed<G>(h.w);
        keep_packed<G>(h.bias);
        #pragma unroll
        for (int m = 0; m < NM; m++) keep_packed<G>(h.tm[m]);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// K slice s of a mix, as MFMA operand fragments.
template <int G, bool Q8, int QS>
__device__ __forceinline__ void mix_fragments(const char* mix, int s, int lane, kr_half8 (&av)[QS]) {
    const char* p = mix + (lane & 15) * kMixPitch<G, Q8> + s * QS * 64 + (lane >> 4) * 16;
    #pragma unroll
    for (int q = 0; q < QS; q++) av[q] = *reinterpret_cast<const kr_half8*>(p + 64 * q);
}

template <bool I8, int QS>
__device__ __forceinline__ void slice_chain(const kr_half8 (&b)[QS], const kr_half8 (&av)[QS], float* dst) {
    if constexpr (I8) {
        kr_int4 acc = kr_int4{0, 0, 0, 0};
        #pragma unroll
        for (int q = 0; q < QS; q++)
            acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(as_i4(b[q]), as_i4(av[q]), acc, 0, 0, 0);
        *reinterpret_cast<kr_int4*>(dst) = acc;
    } else {
        kr_float4 acc = kr_float4{0.f, 0.f, 0.f, 0.f};
        #pragma unroll
        for (int q = 0; q < QS; q++)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[q], av[q], acc, 0, 0, 0);
        *reinterpret_cast<kr_float4*>(dst) = acc;
    }
}

// Slice partials (stride floats apart) folded in order; int8 dequantised.
template <bool I8>
__device__ __forceinline__ kr_float4 fold_slices(const float* p, int S, int stride, float sa, kr_float4 sw) {
    if constexpr (I8) {
        kr_int4 iv = *reinterpret_cast<const kr_int4*>(p);
        for (int q = 1; q < S; q++) iv = iv + *reinterpret_cast<const kr_int4*>(p + q * stride);
        kr_float4 v;
        #pragma unroll
        for (int e = 0; e < 4; e++) v[e] = __fmul_rn(__fmul_rn((float)iv[e], sa), sw[e]);
        return v;
    } else {
        kr_float4 v = *reinterpret_cast<const kr_float4*>(p);
        for (int q = 1; q < S; q++) v = v + *reinterpret_cast<const kr_float4*>(p + q * stride);
        return v;
    }
}

// ---------------------------------------------------------------------------
// LN1-mix, K, V, R and WKV: 16 rows x 16 NS columns of all three products per
// workgroup, wave (j, s) runs K slice s of product j.
// ---------------------------------------------------------------------------
template <int S, int NS, bool I8>
__global__ void __launch_bounds__(192 * S) ln_kvr_wkv_kernel(kr_step_kvr a) {
    constexpr int C = 256 * S, NW = 3 * S, RPW = (16 + NW - 1) / NW, QS = I8 ? 4 : 8;
    constexpr int KB = S * QS, ng = C / (16 * NS);
    static_assert(ng % 8 == 0 && NS <= NW, "a column group's row tiles share an XCD");
    __shared__ __attribute__((aligned(16))) char mix[3 * 16 * kMixPitch<S, I8>];
    __shared__ __attribute__((aligned(16))) float part[3 * S * NS * 256];
    __shared__ float sc[3 * 16];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int j = wave / S, s = wave % S;
    const int n_g = (int)blockIdx.x % ng, m0 = (int)blockIdx.x / ng * 16, n0 = n_g * 16 * NS;
    LnHeld<S, 3, RPW> h;
    ln_request<S, 3, RPW, NW>(a.ln, a.ln.tm, m0, a.M, wave, lane, h);
    __builtin_amdgcn_sched_barrier(0);         // the rows ahead of the weights
    const kr_half* Wf = j == 0 ? a.Wf[0] : (j == 1 ? a.Wf[1] : a.Wf[2]);
    kr_half8 b[NS][QS];
    #pragma unroll
    for (int t = 0; t < NS; t++) {
        const kr_half* bp = Wf + ((size_t)((n0 >> 4) + t) * KB + QS * s) * 512 + lane * 8;
        #pragma unroll
        for (int q = 0; q < QS; q++) b[t][q] = *reinterpret_cast<const kr_half8*>(bp + 512 * q);
    }
    __builtin_amdgcn_sched_barrier(0);
    ln_mix_lds<S, 3, RPW, NW, I8>(h, n_g == 0 ? a.ln.pend : nullptr, m0, a.M, wave, lane, mix, sc);
    // WKV operands of the tile this wave will finish (waves 0 .. NS - 1);
    // requested behind the LN, whose registers they take
    const int em = m0 + (lane & 15), en = n0 + 16 * wave + 4 * (lane >> 4);
    const size_t o = (size_t)min(em, a.M - 1) * C + en;
    kr_float4 sa, sb, sp, dw, du, sw[3];
    if (wave < NS) {
        sa = *reinterpret_cast<const kr_float4*>(a.aa + o);
        sb = *reinterpret_cast<const kr_float4*>(a.bb + o);
        sp = *reinterpret_cast<const kr_float4*>(a.pp + o);
        dw = *reinterpret_cast<const kr_float4*>(a.decay + en);
        du = *reinterpret_cast<const kr_float4*>(a.first + en);
        if constexpr (I8) {
            #pragma unroll
            for (int jj = 0; jj < 3; jj++) sw[jj] = *reinterpret_cast<const kr_float4*>(a.sw[jj] + en);
        }
    }
    __syncthreads();
    kr_half8 av[QS];
    mix_fragments<S, I8, QS>(mix + j * 16 * kMixPitch<S, I8>, s, lane, av);
    #pragma unroll
    for (int t = 0; t < NS; t++) slice_chain<I8, QS>(b[t], av, part + ((j * S + s) * NS + t) * 256 + lane * 4);
    __syncthreads();
    if (wave >= NS || em >= a.M) return;
    kr_float4 kvr[3];
    #pragma unroll
    for (int jj = 0; jj < 3; jj++)
        kvr[jj] = fold_slices<I8>(part + (jj * S * NS + wave) * 256 + lane * 4, S, NS * 256,
                                  I8 ? sc[16 * jj + (lane & 15)] : 0.f, sw[jj]);
    kr_half4 ry;
    #pragma unroll
    for (int e = 0; e < 4; e++) {
        const float r = (float)kr_f16(kr_sigmoid_t<I8>((float)kr_f16(kvr[2][e])));
        WkvState st{sa[e], sb[e], sp[e]};
        ry[e] = wkv_token<I8>(st, dw[e], du[e], kvr[0][e], kvr[1][e], r);
        sa[e] = st.a;
        sb[e] = st.b;
        sp[e] = st.p;
    }
    *reinterpret_cast<kr_float4*>(a.aa + o) = sa;
    *reinterpret_cast<kr_float4*>(a.bb + o) = sb;
    *reinterpret_cast<kr_float4*>(a.pp + o) = sp;
    *reinterpret_cast<kr_half4*>(a.ry + kr_frag_index(em, en, C)) = ry;
}

// ---------------------------------------------------------------------------
// LN2-mix and the channel mix's R and K products: 16 rows x 16 P NS columns
// of one of them per workgroup, wave (p, s) runs K slice s of the NS panels of
// column part p. TIMED (decode-step timing): waves store their start and end
// times at a.stamps; kernels of their own, since the test of a pointer at the
// start holds up the first loads (0.4 us per launch on MI355X).
// ---------------------------------------------------------------------------
template <int S, int P, int NS, bool I8, bool TIMED>
__global__ void __launch_bounds__(64 * S * P) ln_rk_kernel(kr_step_rk a) {
    constexpr int C = 256 * S, NW = S * P, RPW = (16 + NW - 1) / NW, QS = I8 ? 4 : 8;
    constexpr int KB = S * QS, NP = P * NS, TPW = (NP + NW - 1) / NW;
    static_assert(C / 16 % NP == 0, "a group's columns belong to one product");
    __shared__ __attribute__((aligned(16))) char mix[16 * kMixPitch<S, I8>];
    __shared__ __attribute__((aligned(16))) float part[S * NP * 256];
    __shared__ float sc[16];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const unsigned long long t_start = TIMED ? (unsigned long long)wall_clock64() : 0ull;
    const int p = wave / S, s = wave % S;
    const int ng = (C + a.F) / (16 * NP);
    const int n_g = (int)blockIdx.x % ng, m0 = (int)blockIdx.x / ng * 16;
    const bool isk = n_g >= C / (16 * NP);
    const int nb0 = isk ? n_g * NP - C / 16 : n_g * NP;        // first column block of its product
    const kr_half* const tm[1] = {isk ? a.ln.tm[0] : a.ln.tm[1]};
    LnHeld<S, 1, RPW> h;
    ln_request<S, 1, RPW, NW>(a.ln, tm, m0, a.M, wave, lane, h);
    __builtin_amdgcn_sched_barrier(0);
    const kr_half* Wf = isk ? a.WfK : a.WfR;
    kr_half8 b[NS][QS];
    #pragma unroll
    for (int t = 0; t < NS; t++) {
        const kr_half* bp = Wf + ((size_t)(nb0 + p * NS + t) * KB + QS * s) * 512 + lane * 8;
        #pragma unroll
        for (int q = 0; q < QS; q++) b[t][q] = *reinterpret_cast<const kr_half8*>(bp + 512 * q);
    }
    const float* swp = isk ? a.swK : a.swR;
    kr_float4 sw[TPW];
    if constexpr (I8) {
        #pragma unroll
        for (int e = 0; e < TPW; e++)
            sw[e] = *reinterpret_cast<const kr_float4*>(swp + 16 * (nb0 + min(wave + e * NW, NP - 1)) +
                                                        4 * (lane >> 4));
    }
    __builtin_amdgcn_sched_barrier(0);
    ln_mix_lds<S, 1, RPW, NW, I8>(h, n_g == 0 ? a.ln.pend : nullptr, m0, a.M, wave, lane, mix, sc);
    __syncthreads();
    kr_half8 av[QS];
    mix_fragments<S, I8, QS>(mix, s, lane, av);
    #pragma unroll
    for (int t = 0; t < NS; t++) slice_chain<I8, QS>(b[t], av, part + (s * NP + p * NS + t) * 256 + lane * 4);
    __syncthreads();
    const int m = m0 + (lane & 15);
    if (m >= a.M) return;
    #pragma unroll
    for (int e = 0; e < TPW; e++) {
        const int t = wave + e * NW;
        if (t >= NP) break;
        const kr_float4 v = fold_slices<I8>(part + t * 256 + lane * 4, S, NP * 256,
                                            I8 ? sc[lane & 15] : 0.f, sw[e]);
        const int n = 16 * (nb0 + t) + 4 * (lane >> 4);
        kr_half4 y;
        #pragma unroll
        for (int r = 0; r < 4; r++) {
            const float x = (float)kr_f16(v[r]);
            if (isk) {
                const float rr = x > 0.0f ? x : 0.0f;
                y[r] = kr_f16(rr * rr);
            } else {
                y[r] = kr_f16(kr_sigmoid_t<I8>(x));
            }
        }
        if (isk) *reinterpret_cast<kr_half4*>(a.kf + kr_frag_index(m, n, a.F)) = y;
        else *reinterpret_cast<kr_half4*>(a.rf + (size_t)m * C + n) = y;
    }
    if (TIMED && lane == 0) {          // lane 0's row always exists
        unsigned long long* st = a.stamps + 2 * (KR_STAMP_WAVES * blockIdx.x + wave);
        st[0] = t_start;
        st[1] = (unsigned long long)wall_clock64();
    }
}

template <int S, bool I8>
int launch_kvr(const kr_step_kvr& a, hipStream_t s) {
    const int mt = (a.M + 15) / 16, ng = 16 * S;
    // one column panel per workgroup while that fits one round of the 256 CUs
    if (mt * ng <= 256) ln_kvr_wkv_kernel<S, 1, I8><<<mt * ng, 192 * S, 0, s>>>(a);
    else ln_kvr_wkv_kernel<S, 2, I8><<<mt * ng / 2, 192 * S, 0, s>>>(a);
    KR_LAUNCHED();
    return KR_OK;
}

template <int S, int P, int NS, bool I8>
int launch_rk_shape(kr_step_rk a, int blocks, hipStream_t s) {
    const kr_panel_timing tm = kr_gemm_take_timing(blocks, S * P);
    a.stamps = tm.stamps;
    if (tm.start)
        hipExtLaunchKernelGGL((ln_rk_kernel<S, P, NS, I8, true>), dim3(blocks), dim3(64 * S * P), 0u,
                              s, tm.start, tm.stop, 0u, a);
    else if (tm.stamps)
        ln_rk_kernel<S, P, NS, I8, true><<<blocks, 64 * S * P, 0, s>>>(a);
    else
        ln_rk_kernel<S, P, NS, I8, false><<<blocks, 64 * S * P, 0, s>>>(a);
    KR_LAUNCHED();
    return KR_OK;
}

template <int S, bool I8>
int launch_rk(const kr_step_rk& a, hipStream_t s) {
    const int mt = (a.M + 15) / 16, panels = (256 * S + a.F) / 16, rows = std::min(a.M, 16);
    // P waves per slice so that a wave has at most `held` rows to run (int8
    // rows quantise as well), then the fewest panels per workgroup that fit one
    // round of the 256 CUs. Measured on MI355X (decode step, us, C = 768,
    // P = 1 / 2 / 4): fp16 4 rows 302 / 301 / -, 6 rows 303 / 307 / -,
    // 10 rows 343 / 334 / 350, 16 rows 357 / 345 / 352; w8a8 4 rows 315 / 309 /
    // -, 8 rows 346 / 338 / 333, 16 rows 398 / 380 / 374.
    constexpr int held = I8 ? 1 : 3;
    int P = rows > 2 * held * S ? 4 : (rows > held * S ? 2 : 1);
    while (P < 4 && mt * panels / P > 256) P *= 2;
    const int blocks = mt * panels / P;
    if (P == 1) return launch_rk_shape<S, 1, 1, I8>(a, blocks, s);
    if (P == 2) return launch_rk_shape<S, 2, 1, I8>(a, blocks, s);
    if (blocks <= 256) return launch_rk_shape<S, 4, 1, I8>(a, blocks, s);
    return launch_rk_shape<S, 4, 2, I8>(a, blocks / 2, s);
}

// The panel product of one job, one row block per workgroup, and a row copy.
// Bound by the launch chain and the L2 requests in flight, as all panel
// products. One job only: to select one of kr_gemm_multi's three costs scalar
// loads that wait for each other (measured on MI355X, one step of 12 layers, us,
// C = 768, gemm_panel_kernel with the copy in it / this: 1 stream 218 / 212, 128
// streams 322 / 313; w8a8, 128, 362 / 352).
struct kr_gemm_one {
    kr_gemm_args job[1];
    int ep[1];
    int tiles[1];
    unsigned long long* stamps;
};

template <int NS, int MAXT, bool Q8>
__global__ void __launch_bounds__(MAXT) gemm_panel_copy_kernel(kr_gemm_one mj, kr_row_copy copy) {
    panel_product<1, NS, true, Q8, Q8, true>(mj, copy);
}

template <int NS, int MAXT, bool Q8>
int launch_product(const kr_gemm_args& g, int ep, const kr_row_copy& copy, hipStream_t s) {
    const int S = g.K / kKS, blocks = (g.M + 15) / 16 * ((g.N + 16 * NS - 1) / (16 * NS));
    size_t lds = S > 1 ? (size_t)S * NS * 256 * sizeof(float) : 0;
    if (Q8 && S > 1) lds += (size_t)S * 16 * sizeof(float);
    const kr_panel_timing tm = kr_gemm_take_timing(blocks, S);
    const kr_gemm_one mj{{g}, {ep}, {blocks}, tm.stamps};
    if (tm.start)
        hipExtLaunchKernelGGL((gemm_panel_copy_kernel<NS, MAXT, Q8>), dim3(blocks), dim3(64 * S),
                              (uint32_t)lds, s, tm.start, tm.stop, 0u, mj, copy);
    else
        gemm_panel_copy_kernel<NS, MAXT, Q8><<<blocks, 64 * S, lds, s>>>(mj, copy);
    KR_LAUNCHED();
    return KR_OK;
}

template <bool Q8>
int launch_product(const kr_gemm_args& g, int ep, const kr_row_copy& copy, hipStream_t s) {
    // one column panel per workgroup while that fits one round of the 256 CUs,
    // as kr_gemm.hip's busiest-CU model has it at one row block
    const int S = g.K / kKS;
    const bool one = (g.M + 15) / 16 * ((g.N + 15) / 16) <= 256;
    if (S <= 4) return one ? launch_product<1, 256, Q8>(g, ep, copy, s) : launch_product<2, 256, Q8>(g, ep, copy, s);
    if (S <= 12) return one ? launch_product<1, 768, Q8>(g, ep, copy, s) : launch_product<2, 768, Q8>(g, ep, copy, s);
    return one ? launch_product<1, 1024, Q8>(g, ep, copy, s) : launch_product<2, 1024, Q8>(g, ep, copy, s);
}

}  // namespace

int kr_step_launch_kvr(int C, bool i8, const kr_step_kvr& a, hipStream_t s) {
    switch (C / 256) {
        case 1: return i8 ? launch_kvr<1, true>(a, s) : launch_kvr<1, false>(a, s);
        case 2: return i8 ? launch_kvr<2, true>(a, s) : launch_kvr<2, false>(a, s);
        case 3: return i8 ? launch_kvr<3, true>(a, s) : launch_kvr<3, false>(a, s);
        case 4: return i8 ? launch_kvr<4, true>(a, s) : launch_kvr<4, false>(a, s);
        default: return kr_fail(KR_EUNSUPPORTED, "C=%d unsupported (256..1024, step 256)", C);
    }
}

int kr_step_launch_rk(int C, bool i8, const kr_step_rk& a, hipStream_t s) {
    switch (C / 256) {
        case 1: return i8 ? launch_rk<1, true>(a, s) : launch_rk<1, false>(a, s);
        case 2: return i8 ? launch_rk<2, true>(a, s) : launch_rk<2, false>(a, s);
        case 3: return i8 ? launch_rk<3, true>(a, s) : launch_rk<3, false>(a, s);
        case 4: return i8 ? launch_rk<4, true>(a, s) : launch_rk<4, false>(a, s);
        default: return kr_fail(KR_EUNSUPPORTED, "C=%d unsupported (256..1024, step 256)", C);
    }
}

int kr_step_launch_product(const kr_gemm_args& g, int epilogue, const kr_row_copy& copy, hipStream_t s) {
    const int rc = kr_gemm_check(g, epilogue);
    if (rc) return rc;
    KR_REQUIRE(g.a_frag && !g.i8 == !g.a_q16, "step: the product needs fp16 fragment-packed rows");
    KR_REQUIRE(g.M >= 1 && g.M <= KR_GEMM_SMALL_M && g.N < KR_GEMM_SMALL_MAX_N && g.K / kKS <= 16,
               "step: product of M=%d N=%d K=%d", g.M, g.N, g.K);
    return g.i8 ? launch_product<true>(g, epilogue, copy, s) : launch_product<false>(g, epilogue, copy, s);
}
