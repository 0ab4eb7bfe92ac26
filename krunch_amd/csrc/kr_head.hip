// The head (logits = fp16(LN_out(x) @ head)) for more rows than the decode
// step's kernel takes: 256 rows per workgroup held in registers, the weights
// streamed past them. A file of its own: kernels added to kr_gemm.hip move the
// decode step's panel kernels.
#include <algorithm>
#include <type_traits>

#include "kr_gemm.h"

namespace {

// ---------------------------------------------------------------------------
// A workgroup of four waves (one per SIMD, 512 registers each) keeps the whole
// K of its 256 rows as MFMA operands (K = 768: 384 registers) and takes one
// contiguous run of 16-column weight blocks, 24 KB each, through a ring of six
// LDS stages filled by asynchronous copies. Per block a wave multiplies all of
// it with its 64 rows: 96 MFMAs for K = 768, fed by 24 LDS reads, so a CU
// takes 24 KB of operands per 6.3 MMAC where a 256 x 256 tile takes 64 KB per
// 4.2 MMAC K step. One wave per SIMD hides nothing by itself, so the loop is
// pipelined by hand: the fragments of the next group (of the next block, at
// the end) are read while one is multiplied, and a block's results are rounded
// and stored between the next block's MFMAs.
//
// The row groups of one column run are workgroups b, b + 8, ..., on one XCD,
// whose L2 fetches each weight block once for all of them.
//
// Stores are 8 bytes per lane at any row stride (logits rows of 50277 columns
// start at odd multiples of 2 bytes; 2-byte stores there cost two thirds as
// much again as the product).
//
// Bound: at 1024 rows a block takes 1.5 us, about 1.0 of it MFMA issue and the
// rest LDS reads and barriers nothing overlaps; at 8192 the output's 32-byte
// pieces as well (579 us without the stores). Measured on MI355X against the
// 256 x 256 kernel, us, V = 50277, K = 768, rows 50280 / 50277 apart: M = 528
// 76 / 111 -> 67 / 68, 784 110 / 182 -> 83 / 82, 1024 109 / 181 -> 83 / 85,
// 2048 188 / 315 -> 166 / 180, 4096 349 / 562 -> 333 / 356, 8192 714 / 1085
// -> 667 / 692.
// Contract: one MFMA chain over K from zero per output (kr_gemm.h, the head).
// ---------------------------------------------------------------------------
constexpr int kStages = 6;

typedef kr_half4 kr_half4_any __attribute__((aligned(2)));   // any row stride: global memory takes it

// 16-byte asynchronous copy global -> LDS (lane l writes lds + 16 l),
// invisible to the compiler's wait counts.
__device__ __forceinline__ void head_copy(const void* src, unsigned lds) {
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off"
                 :: "s"(lds), "v"(src) : "memory", "m0");
}
template <int N>
__device__ __forceinline__ void wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory");
}

template <int KB>   // K / 32: 8, 16 or 24
__global__ void __launch_bounds__(256, 1) gemm_head_rows_kernel(
        const kr_half* __restrict__ Af, const kr_half* __restrict__ Wf, kr_half* __restrict__ out,
        long long ldo, int M, int N, int mh) {
    constexpr int CPW = KB / 4, NG = KB / 4;          // copies per wave and block; groups of 4 fragments
    constexpr int AHEAD = (kStages - 3) * CPW;        // copies of blocks j + 2 .. j + 4
    __shared__ __attribute__((aligned(1024))) kr_half8 ring[kStages * KB * 64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int nb_total = (N + 15) >> 4;
    const int bx = blockIdx.x, ncr = (int)gridDim.x / mh;
    int h, cr;
    if ((ncr & 7) == 0) {
        h = (bx >> 3) % mh;
        cr = (bx / (8 * mh)) * 8 + (bx & 7);
    } else {
        h = bx % mh;
        cr = bx / mh;
    }
    const int b0 = (int)(((long long)cr * nb_total) / ncr);
    const int nblk = (int)(((long long)(cr + 1) * nb_total) / ncr) - b0;
    const int last_mb = (M - 1) >> 4;
    const int mb0 = 16 * h + 4 * wave;                // row blocks past the last one repeat it
    const bool active = mb0 <= last_mb;
    kr_half8 a[4][KB];
    if (active) {
        #pragma unroll
        for (int i = 0; i < 4; i++) {
            const size_t blk = (size_t)min(mb0 + i, last_mb) * KB;
            #pragma unroll
            for (int q = 0; q < KB; q++)
                a[i][q] = *reinterpret_cast<const kr_half8*>(Af + (blk + q) * 512 + lane * 8);
        }
    }
    const unsigned ring_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)ring;
    auto issue = [&](int j) {
        const char* src = reinterpret_cast<const char*>(
            Wf + ((size_t)(b0 + j) * KB + (size_t)wave * CPW) * 512 + lane * 8);
        const unsigned dst = ring_base + (unsigned)(((j % kStages) * KB + wave * CPW) * 1024);
        #pragma unroll
        for (int u = 0; u < CPW; u++) head_copy(src + u * 1024, dst + u * 1024);
    };
    #pragma unroll
    for (int j = 0; j < kStages - 1; j++)
        if (j < nblk) issue(j);
    wait_vm<0>();
    __syncthreads();
    kr_half8 w[2][4];
    if (active) {
        #pragma unroll
        for (int q = 0; q < 4; q++) w[0][q] = ring[q * 64 + lane];
    }
    // whole: all of the wave's rows exist, so every block but N's last ends in
    // exactly four stores
    const bool whole = active && 16 * (mb0 + 4) <= M;
    const int r = lane & 15, c4 = 4 * (lane >> 4);
    unsigned off[4];
    #pragma unroll
    for (int i = 0; i < 4; i++) off[i] = (unsigned)((16 * i + r) * ldo) + (unsigned)c4;
    kr_half* const rows = out + (size_t)(16 * mb0) * (size_t)ldo;
    kr_float4 prev[4];
    auto round4 = [&](kr_float4 v) {
        kr_half4 x;
        #pragma unroll
        for (int e = 0; e < 4; e++) x[e] = kr_f16(v[e]);
        return x;
    };
    auto store_whole = [&](int j) {
        kr_half* p = rows + 16 * (b0 + j);
        #pragma unroll
        for (int i = 0; i < 4; i++) *reinterpret_cast<kr_half4_any*>(p + off[i]) = round4(prev[i]);
    };
    auto store_edge = [&](int j) {
        const int n = 16 * (b0 + j) + c4;
        #pragma unroll
        for (int i = 0; i < 4; i++) {
            if (16 * (mb0 + i) + r >= M) continue;
            const kr_half4 x = round4(prev[i]);
            kr_half* p = rows + 16 * (b0 + j) + off[i];
            if (n + 3 < N) {
                *reinterpret_cast<kr_half4_any*>(p) = x;
            } else {
                #pragma unroll
                for (int e = 0; e < 4; e++)
                    if (n + e < N) p[e] = x[e];
            }
        }
    };
    // block j: its first group is in w[0]; stores block j - 1's results (STORE)
    auto block = [&](int j, auto store) {
        constexpr bool STORE = decltype(store)::value;
        const kr_half8* st = ring + (j % kStages) * KB * 64;
        const kr_half8* nx = ring + ((j + 1) % kStages) * KB * 64;
        kr_float4 tot[4];
        #pragma unroll
        for (int i = 0; i < 4; i++) tot[i] = kr_float4{0.f, 0.f, 0.f, 0.f};
        #pragma unroll
        for (int g = 0; g < NG; g++) {
            // past the run's last block this reads a stale stage, unused
            const kr_half8* src = g + 1 < NG ? st + 4 * (g + 1) * 64 : nx;
            #pragma unroll
            for (int q = 0; q < 4; q++) w[(g + 1) & 1][q] = src[q * 64 + lane];
            __builtin_amdgcn_sched_barrier(0);
            #pragma unroll
            for (int q = 0; q < 4; q++)
                #pragma unroll
                for (int i = 0; i < 4; i++)
                    tot[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[g & 1][q], a[i][4 * g + q], tot[i],
                                                                    0, 0, 0);
            if constexpr (STORE) {
                if (g == 0) {
                    store_whole(j - 1);
                    #pragma unroll
                    for (int u = 0; u < 16; u++) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
                        __builtin_amdgcn_sched_group_barrier(0x040, 1, 0);
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        #pragma unroll
        for (int i = 0; i < 4; i++) prev[i] = tot[i];
    };
    static_assert(NG % 2 == 0, "a block ends with the next one's first group in w[0]");
    for (int j = 0; j < nblk; j++) {
        // This wave's copies of block j + 1 have landed: those of j + 2 .. j + 4
        // may be in flight, and, issued after them, four stores in each of the
        // last four iterations.
        if (j + kStages - 2 < nblk) {
            if (whole && j >= kStages - 1) wait_vm<AHEAD + 16>();
            else wait_vm<AHEAD>();
        } else {
            wait_vm<0>();
        }
        __syncthreads();   // block j + 1 is in; every wave is done with block j - 1
        if (j + kStages - 1 < nblk) issue(j + kStages - 1);
        if (!active) continue;
        if (whole && j > 0) {
            block(j, std::true_type{});
        } else {
            if (j > 0) store_edge(j - 1);
            block(j, std::false_type{});
        }
    }
    if (active && nblk > 0) store_edge(nblk - 1);
}

}  // namespace

namespace {

// one workgroup per CU: as many column runs (whole eights) as the row groups
// leave; more than 32 row groups go in several launches
constexpr int kLaunchRows = 32 * 256;

int column_runs(int row_groups, int N) {
    const int nb = (N + 15) / 16, most = 256 / row_groups;
    const int n = nb < most ? nb : most;
    return n >= 8 ? n & ~7 : n;
}

}  // namespace

bool kr_gemm_head_rows_ok(int M, int N, int K, long long ldo) {
    return M > 512 && N >= 1 && (K == 256 || K == 512 || K == 768) && ldo >= N && ldo < (1ll << 24);
}

// Where the 256 x 256 kernel stores 2 bytes at a time this one is faster, but
// for few columns over several launches (V = 1000, odd stride, K = 768, 12288
// rows 1.09 of its time). Where it stores 8 (stride and start multiples of
// them), measured on MI355X as this kernel's time over its:
//  * strides of whole 4096 bytes put the 16 rows of a store instruction on one
//    memory channel: V = 65536, M = 1024 0.84..0.89, 1280 0.87..1.47, 2048
//    1.7..2.6, 8192 1.9..2.2;
//  * few columns share the load of the rows among few blocks: V = 1000, M =
//    4096 0.80, 8192 1.02..1.08, 16384 1.4..1.6;
//  * K = 256 and 512, whose rows hold fewer MFMAs per output: once the output
//    outgrows the memory-side cache its partial lines cost memory time (V =
//    50277, K = 256, M = 2048 0.74, 3072 1.43; K = 512, 2048 0.86..1.02, 4096
//    1.11); K = 768 hides that (8192 0.90);
//  * the longest column run against the rounds of 256 x 256 tiles, each about
//    21.5 blocks of 16 columns long, the load of the rows 8: K = 768, V = 50277,
//    M = 1280 (74 blocks, 4 rounds) 0.88, 6144 (401, 19) 0.96, 2816 (205, 9) 1.04,
//    5120 (20 row groups leave 8 runs and 96 CUs idle: 401, 16) 1.10; V = 5000,
//    2048 (18, 1) 0.88, 3072 (28, 1) 1.21, 4096 (28, 2) 0.81, 6144 (48, 2) 1.16;
//  * several launches, at 19: K = 768, V = 20000, M = 16384 (330, 20) 0.95, 12544
//    (330, 16) 1.06..1.10; V = 5000, 9216 (61, 3) 1.10.
bool kr_gemm_head_rows_faster(int M, int N, int K, const kr_half* out, long long ldo) {
    if ((ldo & 3) != 0 || ((uintptr_t)out & 7) != 0) return M <= kLaunchRows || N >= 4096;
    if ((2 * ldo) % 4096 == 0) return M <= 1024;
    if (N < 4096 && M > 4096) return false;
    if (K < 768 && 2ll * M * ldo > 200000000ll) return false;
    if (M > kLaunchRows && !(K == 768 && N >= 20000)) return false;
    const long long tiles = ((M + 255ll) / 256) * ((N + 255) / 256);
    long long blocks = 0;
    for (int r0 = 0; r0 < M; r0 += kLaunchRows) {
        const int runs = column_runs((std::min(M - r0, kLaunchRows) + 255) / 256, N);
        blocks += ((N + 15) / 16 + runs - 1) / runs + 8;
    }
    return 2 * blocks <= (M > kLaunchRows ? 38 : 43) * ((tiles + 255) / 256);
}

int kr_gemm_head_rows(const kr_half* Af, const kr_half* Wf, int M, int N, int K, kr_half* out,
                      long long ldo, hipStream_t s) {
    KR_REQUIRE(Af && Wf && out, "head: null pointer");
    KR_REQUIRE(kr_gemm_head_rows_ok(M, N, K, ldo), "head: unsupported M=%d N=%d K=%d ldo=%lld", M, N, K, ldo);
    KR_REQUIRE(((uintptr_t)Af & 15) == 0 && ((uintptr_t)Wf & 15) == 0,
               "head: operands must be 16-byte aligned");
    for (int r0 = 0; r0 < M; r0 += kLaunchRows) {
        const int m = M - r0 < kLaunchRows ? M - r0 : kLaunchRows, mh = (m + 255) / 256;
        const int ncr = column_runs(mh, N);
        const kr_half* A = Af + (size_t)r0 * K;
        kr_half* o = out + (size_t)r0 * (size_t)ldo;
        switch (K) {
            case 256: gemm_head_rows_kernel<8><<<ncr * mh, 256, 0, s>>>(A, Wf, o, ldo, m, N, mh); break;
            case 512: gemm_head_rows_kernel<16><<<ncr * mh, 256, 0, s>>>(A, Wf, o, ldo, m, N, mh); break;
            default: gemm_head_rows_kernel<24><<<ncr * mh, 256, 0, s>>>(A, Wf, o, ldo, m, N, mh); break;
        }
        KR_LAUNCHED();
    }
    return KR_OK;
}
