// Register-fed GEMM on fragment-packed operands for products of a few hundred
// to a few thousand rows: one short text, the last windows of a file, a
// mid-sized layer call. A file of its own, as kr_wide.hip: kernels added to
// kr_gemm.hip move the decode step's panel kernels.
#include <algorithm>
#include <type_traits>

#include "kr_gemm.h"
#include "kr_gemm_epilogue.h"
#include "kr_math.h"

// ---------------------------------------------------------------------------
// One workgroup of four waves (one per SIMD) takes (16 TM) x (16 TN) output
// tiles. Wave w of round r runs the MFMA chains of K slice 4 r + w over the
// whole tile, its operands straight from memory in registers: 1 KB contiguous
// per load, and as soon as the 32-wide k block q of a slice is consumed, block
// q of the wave's next slice (of this tile or the next one) is requested into
// the same registers. So a wave keeps a slice of operands, up to 64 KB, in
// flight. The four partials of a round meet in LDS, each wave folds its share
// of the tile in slice order, and the barrier waits for LDS only. Persistent:
// one workgroup per CU walks the tiles of up to three products that share M
// and K, the loads running on across tiles and products.
//
// Why: at these sizes a CU gets one to three tiles, and its time is the
// latency and rate of its operand loads. Copies into LDS (kr_gemm.hip's
// rings) deliver ~35-42 GB/s per CU however many are in flight, loads into
// registers about twice that.
// Bound: operand delivery (the K = 3072 product at 777 rows reads 688 KB per
// CU in 14.7 us, 47 GB/s). Measured on MI355X, one layer, us, against
// the 64 x 64 tile kernel on row-major operands (separate launches): fp16 at
// M = 520 / 777 / 1000 / 1300 / 2000 / 2400 rows 127.9 / 138.0 / 145.2 /
// 134.1 / 151.9 / 163.6 -> 70.3 / 90.0 / 103.7 / 92.3 / 142.1 / 163.3 (the
// one-stream sizes include 27-34 us of WKV), w8a8 115.7 / 127.2 / 135.7 /
// 113.3 / 127.7 -> 74.8 / 96.6 / 111.3 / 95.3 / 135.9.
// Reduction contract: kr_gemm.h (256-wide slices folded in order; int8 exact).
// ---------------------------------------------------------------------------
namespace {

struct MidTile {
    int j, m0, n0;      // job, first row block, first column block (16 each)
};

// Virtual block vb -> tile: XCD vb % 8 takes the vb % 8-th contiguous eighth
// of the tile list (the jobs in order, rows fastest), so the column groups of
// an XCD, and with them the weight panels its L2 holds, are few.
template <int TM, int TN>
__device__ __forceinline__ bool mid_tile(const kr_gemm_multi& mj, int vb, int total, MidTile& t) {
    const int per = (total + 7) / 8;
    if ((vb >> 3) >= per) return false;
    int r = __builtin_amdgcn_readfirstlane((vb & 7) * per + (vb >> 3));
    if (r >= total) return false;
    t.j = 0;
    while (r >= mj.tiles[t.j]) r -= mj.tiles[t.j++];
    const int gy = (mj.job[0].M + 16 * TM - 1) / (16 * TM);
    t.m0 = r % gy * TM;
    t.n0 = r / gy * TN;
    return true;
}

// The kernel's first argument where it lies: a job's fields at a run-time
// index are then scalar loads (an indexed by-value argument is copied to
// scratch memory).
__device__ __forceinline__ const kr_gemm_multi& kernarg_jobs() {
    return *(const kr_gemm_multi*)__builtin_amdgcn_kernarg_segment_ptr();
}

__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <bool I8, int TM, int TN>
__global__ void __launch_bounds__(256, 1) gemm_mid_kernel(kr_gemm_multi, int total) {
    constexpr int QS = I8 ? 4 : 8;                 // 1 KB blocks per 256-wide slice and fragment row
    constexpr int TT = TM * TN, PW = (TT + 3) / 4; // tiles folded per wave
    typedef typename std::conditional<I8, kr_int4, kr_float4>::type Acc;
    __shared__ __attribute__((aligned(16))) Acc part[2][4][TT * 64];
    const kr_gemm_multi& mj = kernarg_jobs();
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int G = gridDim.x, M = mj.job[0].M, K = mj.job[0].K;
    const int S = K / KR_GEMM_KSPLIT, R = (S + 3) / 4, KB = S * QS;
    const int last_mb = (M - 1) >> 4;

    MidTile cur;
    int vb = blockIdx.x;
    if (!mid_tile<TM, TN>(mj, vb, total, cur)) return;

    // operand blocks of (tile t, slice s): row block i at pa[i], column block at pw[i]
    const kr_half* pa[TM];
    const kr_half* pw[TN];
    auto sources = [&](const MidTile& t, int s) {
        const kr_gemm_args& g = mj.job[t.j];
        const int last_nb = (g.N - 1) >> 4;
        // blocks past the last row or column block repeat it (never stored)
        #pragma unroll
        for (int i = 0; i < TM; i++)
            pa[i] = g.A + ((size_t)min(t.m0 + i, last_mb) * KB + s * QS) * 512;
        #pragma unroll
        for (int i = 0; i < TN; i++)
            pw[i] = g.Wf + ((size_t)min(t.n0 + i, last_nb) * KB + s * QS) * 512;
    };
    kr_half8 a[QS][TM], w[QS][TN];
    auto load = [&](int q) {
        #pragma unroll
        for (int i = 0; i < TN; i++) w[q][i] = *reinterpret_cast<const kr_half8*>(pw[i] + q * 512 + lane * 8);
        #pragma unroll
        for (int i = 0; i < TM; i++) a[q][i] = *reinterpret_cast<const kr_half8*>(pa[i] + q * 512 + lane * 8);
    };
    // The chains of the slice held, the next slice requested behind them (or
    // not, after the last one: a body of its own, since a conditional load
    // makes the compiler wait as if it had not been issued, for all of them).
    auto chains = [&](Acc (&acc)[TM][TN], auto more) {
        #pragma unroll
        for (int i = 0; i < TM; i++)
            #pragma unroll
            for (int t = 0; t < TN; t++) acc[i][t] = Acc{0, 0, 0, 0};
        #pragma unroll
        for (int q = 0; q < QS; q++) {
            #pragma unroll
            for (int i = 0; i < TM; i++)
                #pragma unroll
                for (int t = 0; t < TN; t++) {
                    if constexpr (I8)
                        acc[i][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(as_i4(w[q][t]), as_i4(a[q][i]),
                                                                         acc[i][t], 0, 0, 0);
                    else
                        acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[q][t], a[q][i], acc[i][t],
                                                                          0, 0, 0);
                }
            if constexpr (decltype(more)::value) load(q);
        }
    };
    const bool works = wave < S;                   // a wave past the slices only folds
    if (works) {
        sources(cur, wave);
        #pragma unroll
        for (int q = 0; q < QS; q++) load(q);
    }
    int buf = 0;
    while (true) {
        MidTile nxt;
        const bool has_next = mid_tile<TM, TN>(mj, vb + G, total, nxt);
        const kr_gemm_args& g = mj.job[cur.j];
        Acc tot[PW];
        for (int r = 0; r < R; r++) {
            const int s = 4 * r + wave;
            if (s < S) {
                // this wave's next slice: the next round's, or the next tile's first
                const bool again = s + 4 < S;
                const bool more = again || has_next;
                if (more) sources(again ? cur : nxt, again ? s + 4 : wave);
                Acc acc[TM][TN];
                if (more) chains(acc, std::true_type{});
                else chains(acc, std::false_type{});
                #pragma unroll
                for (int i = 0; i < TM; i++)
                    #pragma unroll
                    for (int t = 0; t < TN; t++) part[buf][wave][(i * TN + t) * 64 + lane] = acc[i][t];
            }
            lds_barrier();
            // fold this round's slices onto the wave's tiles, in order
            #pragma unroll
            for (int p = 0; p < PW; p++) {
                const int t = wave + 4 * p;
                if (t >= TT) break;
                #pragma unroll
                for (int u = 0; u < 4; u++) {
                    if (4 * r + u >= S) break;
                    const Acc v = part[buf][u][t * 64 + lane];
                    tot[p] = (r | u) == 0 ? v : tot[p] + v;
                }
            }
            buf ^= 1;
        }
        // lane: row 16 (m0 + i) + lane % 16, columns 4 (lane / 16) .. + 3 of block n0 + t
        const int ep = mj.ep[cur.j];
        const uintptr_t ovec = ep == KR_EP_F32 ? 15 : 7;
        const bool vec_ok = (g.ldo & 3) == 0 && ((uintptr_t)g.out & ovec) == 0 &&
                            ((ep != KR_EP_RESID && ep != KR_EP_GATED) || ((uintptr_t)g.res & 7) == 0) &&
                            (ep != KR_EP_GATED || ((uintptr_t)g.gate & 7) == 0);
        auto store = [&](auto epc) {
            constexpr int EP = decltype(epc)::value;
            #pragma unroll
            for (int p = 0; p < PW; p++) {
                const int t = wave + 4 * p;
                if (t >= TT) break;
                const int m = 16 * (cur.m0 + t / TN) + (lane & 15);
                const int n = 16 * (cur.n0 + t % TN) + 4 * (lane >> 4);
                if (m >= M || n >= g.N) continue;
                kr_float4 v;
                if constexpr (I8) {
                    const float sa = g.sa[m];
                    #pragma unroll
                    for (int e = 0; e < 4; e++)
                        v[e] = __fmul_rn(__fmul_rn((float)tot[p][e], sa), g.sw[min(n + e, g.N - 1)]);
                } else {
                    v = tot[p];
                }
                if constexpr (EP == KR_EP_F16 || EP == KR_EP_SIGMOID || EP == KR_EP_RELUSQ) {
                    if (g.out_frag) {   // the [M, N] operand of the next product (N % 32 == 0)
                        kr_gemm_args o = g;
                        o.out = reinterpret_cast<kr_half*>(g.out) + kr_frag_index(m, n, g.N);
                        o.ldo = 0;
                        store_row4<EP, I8>(o, 0, 0, v, true);
                        continue;
                    }
                }
                store_row4<EP, I8>(g, m, n, v, vec_ok && n + 3 < g.N);
            }
        };
        switch (ep) {
            case KR_EP_F32: store(std::integral_constant<int, KR_EP_F32>{}); break;
            case KR_EP_F16: store(std::integral_constant<int, KR_EP_F16>{}); break;
            case KR_EP_SIGMOID: store(std::integral_constant<int, KR_EP_SIGMOID>{}); break;
            case KR_EP_RELUSQ: store(std::integral_constant<int, KR_EP_RELUSQ>{}); break;
            case KR_EP_RESID: store(std::integral_constant<int, KR_EP_RESID>{}); break;
            default: store(std::integral_constant<int, KR_EP_GATED>{}); break;
        }
        if (!has_next) break;
        vb += G;
        cur = nxt;
    }
}

template <bool I8, int TM, int TN>
int launch_mid(kr_gemm_multi mj, hipStream_t s) {
    long long total = 0;
    for (int j = 0; j < mj.njobs; j++) {
        const kr_gemm_args& g = mj.job[j];
        mj.tiles[j] = (int)((long long)((g.M + 16 * TM - 1) / (16 * TM)) * ((g.N + 16 * TN - 1) / (16 * TN)));
        total += mj.tiles[j];
    }
    const int grid = (int)std::min<long long>(256, (total + 7) / 8 * 8);   // one workgroup per CU
    gemm_mid_kernel<I8, TM, TN><<<grid, 256, 0, s>>>(mj, (int)total);
    KR_LAUNCHED();
    return KR_OK;
}

}  // namespace

int kr_gemm_launch_mid(const kr_gemm_multi& mj, hipStream_t s) {
    // tile shape: the fewest operand blocks on the busiest CU (the first of
    // equals). 4 x 4 against the rule's choice, us per layer: 82.3 / 75.2 at
    // M = 600 (2 x 4), 94.1 / 90.0 at 777 (3 x 4), 108.1 / 103.7 at 1000 (4 x 3)
    constexpr int shapes[4][2] = {{4, 4}, {4, 3}, {2, 4}, {3, 4}};
    long long best = -1;
    int bi = 0;
    for (int i = 0; i < 4; i++) {
        const int TM = shapes[i][0], TN = shapes[i][1];
        long long total = 0;
        for (int j = 0; j < mj.njobs; j++)
            total += (long long)((mj.job[j].M + 16 * TM - 1) / (16 * TM)) *
                     ((mj.job[j].N + 16 * TN - 1) / (16 * TN));
        const long long cost = (total + 255) / 256 * (TM + TN);
        if (best < 0 || cost < best) { best = cost; bi = i; }
    }
    if (mj.job[0].i8) {
        if (bi == 0) return launch_mid<true, 4, 4>(mj, s);
        if (bi == 1) return launch_mid<true, 4, 3>(mj, s);
        if (bi == 3) return launch_mid<true, 3, 4>(mj, s);
        return launch_mid<true, 2, 4>(mj, s);
    }
    if (bi == 0) return launch_mid<false, 4, 4>(mj, s);
    if (bi == 1) return launch_mid<false, 4, 3>(mj, s);
    if (bi == 3) return launch_mid<false, 3, 4>(mj, s);
    return launch_mid<false, 2, 4>(mj, s);
}
