// Stepped layer products with their LayerNorm-mix in the same launch (kr_step.hip).
#pragma once
#include "kr_gemm.h"

// Whether a stepped layer of M streams takes them: beyond, the LN that every
// column group repeats (C / 16 groups of C values per row) costs more than the
// launches it saves. Measured on MI355X, one step of 12 layers, F = 4 C, us,
// six launches per layer / four. fp16: C = 256, M = 16 213 / 190, 160 275 / 215;
// 512, 16 267 / 227, 160 346 / 267; 768, 16 291 / 264, 128 369 / 323, 144
// 371 / 373, 160 372 / 378; 1024, 8 330 / 311, 48 352 / 344, 64 382 / 382, 96
// 408 / 437, 128 436 / 531. w8a8, whose rows are quantised as well: C = 256, 12
// 237 / 225, 16 240 / 254, 96 263 / 264, 97 290 / 264 (the panel products'
// tiles change there), 128 301 / 268; 512, 16 302 / 282, 128 354 / 304; 768, 16
// 327 / 320, 128 399 / 353; 1024, 16 361 / 346, 96 422 / 382, 112 436 / 445.
// Decode runs (C = 768): fp16 128 streams 422 / 393, 144 434 / 438; w8a8 128
// 442 / 405, 144 440 / 455. The limits at C <= 512 (fp16) and 512 (w8a8) are the
// last rows measured ahead, not crossovers.
inline bool kr_step_fuse_ok(int C, int M, bool i8) {
    if (i8) return C <= 256 ? M <= 12 || (M > 96 && M <= 128) : M <= (C <= 768 ? 128 : 96);
    return M <= (C <= 512 ? 160 : (C <= 768 ? 128 : 48));
}

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
// The layer's O and V products (one fragment-packed product, w8a8: of fp16 rows
// quantised on load), with the carried rows copied in the same launch.
int kr_step_launch_product(const kr_gemm_args& g, int epilogue, const kr_row_copy& copy, hipStream_t s);
