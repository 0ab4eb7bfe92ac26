// The WKV recurrence (wkv_kernel.cu:52-73 semantics): one token's update,
// shared by the packed kernels (wkv_kernel in kr_layer.hip, kr_wkv.hip) and the
// stepped K, V, R + WKV kernel (kr_layer.hip), and the packed launch.
#pragma once
#include "kr_common.h"
#include "kr_math.h"

namespace {

struct WkvState {
    float a, b, p;
};

// ry = fp16(r * fp16(num / den)), the quotient by codec.
template <bool DET>
__device__ __forceinline__ kr_half wkv_receive(float num, float den, float rr) {
    float y;
    if constexpr (DET) y = num / den;
    else y = num * __builtin_amdgcn_rcpf(den);
    return kr_f16(rr * (float)kr_f16(y));
}

// One token of the recurrence; returns ry.
// DET: exps by kr_kexp and an IEEE division (the w8a8 codec, which the oracle
// restates bit for bit; every exp argument here is <= 0). Otherwise (the fp16
// codec) the hardware exp and the quotient as numerator times the hardware
// reciprocal (~1 ulp; y is rounded to fp16 next): the packed and stepped
// paths both run this function, so their bits agree.
template <bool DET>
__device__ __forceinline__ kr_half wkv_token(WkvState& st, float w, float u, float kk, float vv,
                                             float rr) {
    const float ww = u + kk;
    const float p1 = fmaxf(st.p, ww);
    const float e1 = kr_exp_t<DET>(st.p - p1), e2 = kr_exp_t<DET>(ww - p1);
    const float num = e1 * st.a + e2 * vv, den = e1 * st.b + e2;   // den >= min(1, bb) > 0
    const kr_half ry = wkv_receive<DET>(num, den, rr);
    const float ww2 = w + st.p;
    const float p2 = fmaxf(ww2, kk);
    const float f1 = kr_exp_t<DET>(ww2 - p2), f2 = kr_exp_t<DET>(kk - p2);
    st.a = f1 * st.a + f2 * vv;
    st.b = f1 * st.b + f2;
    st.p = p2;
    return ry;
}

}  // namespace

// WKV over T tokens of B streams, fused with the receptance product:
// ry = fp16(r * fp16(y)). k, v fp32 and r fp16 are [B*T, C]; ry [B*T, C] is
// row-major, or fragment-packed (ry_frag) for the output projection. The
// state aa, bb, pp [B, C] is updated in place.
struct kr_wkv_args {
    const float* k;
    const float* v;
    const kr_half* r;
    const float* decay;        // [C] (already -exp)
    const float* first;        // [C]
    float* aa;
    float* bb;
    float* pp;
    kr_half* ry;
    int B, T, C, ry_frag;
};

// det: kr_kexp and an IEEE division (the w8a8 codec).
int kr_wkv_launch(const kr_wkv_args& a, bool det, hipStream_t s);
// Whether the window goes to the kernel split over time, and its launch (kr_wkv.hip).
bool kr_wkv_use_scan(const kr_wkv_args& a, bool det);
int kr_wkv_launch_scan(const kr_wkv_args& a, bool det, hipStream_t s);
