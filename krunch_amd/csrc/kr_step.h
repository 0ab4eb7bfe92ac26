// Stepped layer products with their LayerNorm-mix in the same launch (kr_step.hip).
#pragma once
#include "kr_gemm.h"

// Streams up to which they are used: beyond, the LN that every column group
// repeats costs more than the launches it saves (figures in kr_step.hip).
#define KR_STEP_FUSE_M 160
#define KR_STEP_FUSE_M_I8 128

struct kr_step_ln {
    const kr_half* x;          // [M, C] residual stream
    const kr_half* ln_w;
    const kr_half* ln_b;
    const kr_half* tm[3];
    const kr_half* state;      // [M, C] carried rows (read)
    kr_half* pend;             // [M, C] the new carried rows: the next product copies them to state
};

struct kr_step_kvr {
    kr_step_ln ln;             // LN1; tm: k, v, r
    const kr_half* Wf[3];      // K, V, R weights, fragment-packed (int8: same bytes)
    const float* sw[3];        // w8a8: per-output-channel scales
    const float* decay;        // [C] (already -exp)
    const float* first;        // [C]
    float* aa;                 // [M, C] WKV state, updated in place
    float* bb;
    float* pp;
    kr_half* ry;               // fragment-packed [M16, C]
    int M;
};

struct kr_step_rk {
    kr_step_ln ln;             // LN2; tm: k, r
    const kr_half* WfR;        // [C, C], [F, C] fragment-packed
    const kr_half* WfK;
    const float* swR;          // w8a8
    const float* swK;
    kr_half* rf;               // [M, C] fp16(sigmoid(fp16(acc)))
    kr_half* kf;               // fragment-packed [M16, F] fp16(relu(fp16(acc))^2)
    int F, M;                  // F % 256 == 0
    unsigned long long* stamps;   // decode-step timing (kr_gemm.h), set by the launch
};

int kr_step_launch_kvr(int C, bool i8, const kr_step_kvr& a, hipStream_t s);
int kr_step_launch_rk(int C, bool i8, const kr_step_rk& a, hipStream_t s);
