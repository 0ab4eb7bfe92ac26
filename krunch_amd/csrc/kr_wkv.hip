// Packed WKV (T tokens per stream) split over time, and the C-ABI entry point.
// wkv_kernel (kr_layer.hip) takes one lane per (stream, channel) and is
// sequential over T. The serial part of the recurrence is only
// p' = max(w + p, k) and a' = f1 a + f2 v, b' = f1 b + f2 (two dependent
// operations per token each); the exponentials and the quotient of a token
// need nothing but its own p, a, b. A workgroup here splits those over waves.
// Same operations and bits as wkv_token (kr_wkv.h).
#include <algorithm>

#include "kr_gemm.h"
#include "kr_wkv.h"
#include "krunch_hip.h"

namespace {

// ---------------------------------------------------------------------------
// 16 channels of one stream per workgroup, the window in chunks of kScanTok
// tokens, five stages one chunk apart (one barrier per chunk):
//   K  (workers)  k of each token into LDS; v, r stay in registers
//   P  (wave 0)   the p chain; leaves p before each token in LDS
//   E  (workers)  f1, f2 v, f2 of each token into LDS; e1, e2, e2 v stay in
//                 registers until the token's Y
//   AB (wave 1)   the a chain in lanes 0..15 and the b chain in lanes 16..31;
//                 a, b before each token replace f2 v, f2
//   Y  (workers)  the quotient and ry
// A worker takes 4 tokens x 16 channels at a time. LDS arrays are [channel]
// [token] with a pitch of kScanTok + 4 words: a chain reads and writes 4
// tokens per instruction (16 lanes on 64 distinct banks), and a worker's 4
// tokens x 16 channels are 64 distinct banks too. The barriers wait for LDS
// only, so the next chunk's global loads stay in flight across them.
// Bound: at few workgroups the latency of a chunk's dependent steps (~0.75 us
// per 32 tokens); with several workgroups per CU the VALU work of the six
// waves, ~1.6 times wkv_kernel's. Measured on MI355X, C = 768 (wkv_kernel ->
// this): B = 1, T = 1000 171 -> 27 us; B = 8, T = 128 23 -> 8; B = 20,
// T = 1024 177 -> 79. Eight workers per workgroup instead of four: 22 us at
// B = 1 but 118 at B = 20. Loads three chunks ahead instead of one: 27 / 109
// (118 registers). [token][channel] arrays and chunks of 64: 38 / 162.
// ---------------------------------------------------------------------------
constexpr int kScanTok = 32, kScanCh = 16, kScanWorkers = 4;
constexpr int kScanSteps = kScanTok / (4 * kScanWorkers);   // token groups of a worker per chunk
constexpr int kScanThreads = 64 * (2 + kScanWorkers);
constexpr int kScanPitch = kScanTok + 4, kScanBuf = kScanPitch * kScanCh;
static_assert(kScanTok % (4 * kScanWorkers) == 0 && kScanTok % 16 == 0, "chunk split");

__device__ __forceinline__ void lds_barrier() {
    __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <bool DET>
__global__ void __launch_bounds__(kScanThreads) wkv_scan_kernel(kr_wkv_args g) {
    __shared__ __attribute__((aligned(16))) float sk[2][kScanBuf];       // k
    __shared__ __attribute__((aligned(16))) float sp[2][kScanBuf];       // p before the token
    __shared__ __attribute__((aligned(16))) float sf[3][3][kScanBuf];    // [slot][f1 | f2 v -> a | f2 -> b]
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int C = g.C, T = g.T, b = blockIdx.y;
    const int ch = lane & 15, c = blockIdx.x * kScanCh + ch;
    const int cc = min(c, C - 1);            // lanes past C compute, never store
    const size_t s = (size_t)b * C + cc;
    const int nc = (T + kScanTok - 1) / kScanTok;

    if (wave == 0) {
        // ---- P: chunk i - 1 in iteration i
        const float w = g.decay[cc];
        float p = g.pp[s];
        for (int i = 0; i < nc + 4; i++) {
            const int j = i - 1;
            if (j >= 0 && j < nc && lane < 16) {
                const kr_float4* in = reinterpret_cast<const kr_float4*>(sk[j & 1] + ch * kScanPitch);
                kr_float4* out = reinterpret_cast<kr_float4*>(sp[j & 1] + ch * kScanPitch);
                const int n = T - j * kScanTok;
                kr_float4 kk[kScanTok / 4];
                #pragma unroll
                for (int q = 0; q < kScanTok / 4; q++) kk[q] = in[q];
                if (n >= kScanTok) {
                    #pragma unroll
                    for (int q = 0; q < kScanTok / 4; q++) {
                        kr_float4 before;
                        #pragma unroll
                        for (int e = 0; e < 4; e++) {
                            before[e] = p;
                            p = fmaxf(w + p, kk[q][e]);
                        }
                        out[q] = before;
                    }
                } else {
                    #pragma unroll
                    for (int q = 0; q < kScanTok / 4; q++) {
                        if (4 * q >= n) break;
                        kr_float4 before;
                        #pragma unroll
                        for (int e = 0; e < 4; e++) {
                            before[e] = p;
                            const float p2 = fmaxf(w + p, kk[q][e]);
                            p = 4 * q + e < n ? p2 : p;
                        }
                        out[q] = before;
                    }
                }
            }
            lds_barrier();
        }
        if (lane < 16 && c < C) g.pp[s] = p;
    } else if (wave == 1) {
        // ---- AB: chunk i - 3 in iteration i
        const bool isb = lane >= 16;
        float* st = isb ? g.bb : g.aa;
        float x = st[s];
        for (int i = 0; i < nc + 4; i++) {
            const int j = i - 3;
            if (j >= 0 && j < nc && lane < 32) {
                const kr_float4* f1 = reinterpret_cast<const kr_float4*>(sf[j % 3][0] + ch * kScanPitch);
                kr_float4* io = reinterpret_cast<kr_float4*>(sf[j % 3][isb ? 2 : 1] + ch * kScanPitch);
                const int n = T - j * kScanTok;
                kr_float4 f[kScanTok / 4], a[kScanTok / 4];
                #pragma unroll
                for (int q = 0; q < kScanTok / 4; q++) { f[q] = f1[q]; a[q] = io[q]; }
                if (n >= kScanTok) {
                    #pragma unroll
                    for (int q = 0; q < kScanTok / 4; q++) {
                        kr_float4 before;
                        #pragma unroll
                        for (int e = 0; e < 4; e++) {
                            before[e] = x;
                            x = f[q][e] * x + a[q][e];
                        }
                        io[q] = before;
                    }
                } else {
                    #pragma unroll
                    for (int q = 0; q < kScanTok / 4; q++) {
                        if (4 * q >= n) break;
                        kr_float4 before;
                        #pragma unroll
                        for (int e = 0; e < 4; e++) {
                            before[e] = x;
                            const float nx = f[q][e] * x + a[q][e];
                            x = 4 * q + e < n ? nx : x;
                        }
                        io[q] = before;
                    }
                }
            }
            lds_barrier();
        }
        if (lane < 32 && c < C) st[s] = x;
    } else {
        // ---- K: chunk i, E: chunk i - 2, Y: chunk i - 4
        const float w = g.decay[cc], u = g.first[cc];
        const int t_in = 4 * (wave - 2) + (lane >> 4);      // + 4 kScanWorkers per step
        // a chunk's rows: a uniform base plus a 32-bit offset inside the chunk
        const size_t stream = (size_t)b * T * C;
        float kn[kScanSteps], vn[kScanSteps];                // the next chunk, in flight
        kr_half rn[kScanSteps];
        struct Raw { float k, v; kr_half r; } raw[2][kScanSteps] = {};
        struct Held { float e1, e2, e2v, r; } held[2][kScanSteps] = {};
        auto load = [&](int i) {
            const size_t row0 = stream + (size_t)i * kScanTok * C;
            const int last = T - 1 - i * kScanTok;           // tokens past T repeat the last one
            #pragma unroll
            for (int q = 0; q < kScanSteps; q++) {
                const unsigned o = (unsigned)(min(t_in + 4 * kScanWorkers * q, last) * C + cc);
                kn[q] = (g.k + row0)[o];
                vn[q] = (g.v + row0)[o];
                rn[q] = (g.r + row0)[o];
            }
        };
        load(0);
        for (int i = 0; i < nc + 4; i++) {
            const int jy = i - 4, je = i - 2;
            if (jy >= 0) {
                const float (*src)[kScanBuf] = sf[jy % 3];
                const int n = T - jy * kScanTok;
                kr_half* rows = g.ry + stream + (size_t)jy * kScanTok * C;
                #pragma unroll
                for (int q = 0; q < kScanSteps; q++) {
                    const int tl = t_in + 4 * kScanWorkers * q;
                    const Held h = held[1][q];
                    const float a = src[1][ch * kScanPitch + tl], bb = src[2][ch * kScanPitch + tl];
                    const float num = h.e1 * a + h.e2v, den = h.e1 * bb + h.e2;
                    const kr_half ry = wkv_receive<DET>(num, den, h.r);
                    if (tl < n && c < C) {
                        if (g.ry_frag)
                            g.ry[kr_frag_index((long long)b * T + jy * kScanTok + tl, c, C)] = ry;
                        else
                            rows[(unsigned)(tl * C + cc)] = ry;
                    }
                }
            }
            #pragma unroll
            for (int q = 0; q < kScanSteps; q++) held[1][q] = held[0][q];
            if (je >= 0 && je < nc) {
                float (*dst)[kScanBuf] = sf[je % 3];
                #pragma unroll
                for (int q = 0; q < kScanSteps; q++) {
                    const int o = ch * kScanPitch + t_in + 4 * kScanWorkers * q;
                    const float p = sp[je & 1][o], kk = raw[1][q].k, vv = raw[1][q].v;
                    const float ww = u + kk, p1 = fmaxf(p, ww);
                    const float ww2 = w + p, p2 = fmaxf(ww2, kk);
                    Held h;
                    h.e1 = kr_exp_t<DET>(p - p1);
                    h.e2 = kr_exp_t<DET>(ww - p1);
                    h.e2v = h.e2 * vv;
                    h.r = (float)raw[1][q].r;
                    held[0][q] = h;
                    const float f2 = kr_exp_t<DET>(kk - p2);
                    dst[0][o] = kr_exp_t<DET>(ww2 - p2);
                    dst[1][o] = f2 * vv;
                    dst[2][o] = f2;
                }
            }
            #pragma unroll
            for (int q = 0; q < kScanSteps; q++) raw[1][q] = raw[0][q];
            if (i < nc) {
                #pragma unroll
                for (int q = 0; q < kScanSteps; q++) {
                    raw[0][q] = Raw{kn[q], vn[q], rn[q]};
                    sk[i & 1][ch * kScanPitch + t_in + 4 * kScanWorkers * q] = kn[q];
                }
                if (i + 1 < nc) load(i + 1);
            }
            lds_barrier();
        }
    }
}

}  // namespace

bool kr_wkv_use_scan(const kr_wkv_args& a, bool det) {
    // The scan kernel up to the stream count where its extra VALU work costs
    // more than wkv_kernel's serial chain. Measured on MI355X at C = 768,
    // T = 1024 (wkv_kernel / scan, us): fp16 B = 20 177 / 79, B = 64 200 / 312
    // (equal near B = 35, 1680 workgroups); w8a8, whose exponentials and
    // division make the chain longer, scan ahead by 146 us per layer at
    // B = 32, by 42 at B = 48, behind by 24 at B = 64. Below 32 tokens
    // (one chunk) its five stages cost more than they hide: B = 64, T = 16
    // 9 / 16 us. At one to two chunks the pipeline's fill is a good part of
    // the run, so the crossover comes earlier: fp16 T = 33, B = 16 / 24 / 32
    // 8.7 / 8.8 / 8.8 (wkv_kernel) against 7.4 / 9.8 / 10.7; w8a8 T = 40, a
    // layer at B = 44 3 us ahead, at B = 53 3 us behind.
    const long long wgs = (long long)a.B * ((a.C + kScanCh - 1) / kScanCh);
    const long long most = a.T < 64 ? (det ? 2048 : 1024) : (det ? 2560 : 1536);
    return a.T >= 32 && wgs <= most;
}

int kr_wkv_launch_scan(const kr_wkv_args& a, bool det, hipStream_t s) {
    const dim3 grid((a.C + kScanCh - 1) / kScanCh, a.B);
    if (det) wkv_scan_kernel<true><<<grid, kScanThreads, 0, s>>>(a);
    else wkv_scan_kernel<false><<<grid, kScanThreads, 0, s>>>(a);
    KR_LAUNCHED();
    return KR_OK;
}

extern "C" int kr_wkv(int B, int T, int C, const float* decay, const float* first, const float* k,
                      const float* v, const uint16_t* r, float* aa, float* bb, float* pp,
                      uint16_t* ry, void* stream) {
    KR_REQUIRE(decay && first && k && v && r && aa && bb && pp && ry, "kr_wkv: null pointer");
    KR_REQUIRE(B >= 1 && T >= 0 && C >= 1, "kr_wkv: bad shape");
    if (T == 0) return KR_OK;
    return kr_wkv_launch(kr_wkv_args{k, v, reinterpret_cast<const kr_half*>(r), decay, first, aa, bb,
                                     pp, reinterpret_cast<kr_half*>(ry), B, T, C, 0},
                         false, kr_stream(stream));
}
