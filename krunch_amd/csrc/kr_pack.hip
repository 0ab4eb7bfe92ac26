// Weight copies for the products: W [K, N] transposed and fragment-packed in
// one launch. A file of its own: kernels added to kr_gemm.hip move the decode
// step's panel kernels.
#include "kr_gemm.h"
#include "krunch_hip.h"

namespace {

// A 32 x 32 tile of W goes through LDS once and leaves as 32 rows of Wt and as
// two 1 KB blocks of the fragment layout (rows of W^T past N: zeros).
// Bound: HBM (a [768, 3072] weight and its two copies, 14 MB). In place of a
// transpose and a pack launch, it is there for the first call on new weights,
// which is host-bound: one launch and one allocation per weight, as without
// the packed copy.
__global__ void __launch_bounds__(256)
transpose_pack_kernel(const kr_half* __restrict__ W, long long ldw, int K, int N,
                      kr_half* __restrict__ Wt, long long ldt, kr_half* __restrict__ Wf) {
    __shared__ kr_half tile[32][33];
    const int k0 = blockIdx.y * 32, n0 = blockIdx.x * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;   // 32 x 8
    for (int r = ty; r < 32; r += 8)
        tile[r][tx] = n0 + tx < N ? W[(size_t)(k0 + r) * ldw + n0 + tx] : (kr_half)0.0f;
    __syncthreads();
    for (int r = ty; r < 32; r += 8)
        if (n0 + r < N) Wt[(size_t)(n0 + r) * ldt + k0 + tx] = tile[tx][r];
    const int rb = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (rb >= 2 || n0 + 16 * rb >= (int)kr_frag_rows(N)) return;
    kr_half8 v;
    #pragma unroll
    for (int e = 0; e < 8; e++) v[e] = tile[8 * (lane >> 4) + e][16 * rb + (lane & 15)];
    const size_t block = ((size_t)(n0 >> 4) + rb) * (size_t)(K >> 5) + (size_t)(k0 >> 5);
    *reinterpret_cast<kr_half8*>(Wf + block * 512 + lane * 8) = v;
}

}  // namespace

extern "C" int kr_transpose_pack_f16(const uint16_t* W, long long ldw, int K, int N, uint16_t* Wt,
                                     long long ldt, uint16_t* Wf, void* stream) {
    KR_REQUIRE(W && Wt && Wf && K >= 32 && K % 32 == 0 && N >= 1 && ldw >= N && ldt >= K,
               "kr_transpose_pack_f16: bad args (K must be a multiple of 32)");
    KR_REQUIRE(((uintptr_t)Wf & 15) == 0, "kr_transpose_pack_f16: Wf must be 16-byte aligned");
    const dim3 grid((N + 31) / 32, K / 32);
    transpose_pack_kernel<<<grid, 256, 0, kr_stream(stream)>>>(
        reinterpret_cast<const kr_half*>(W), ldw, K, N, reinterpret_cast<kr_half*>(Wt), ldt,
        reinterpret_cast<kr_half*>(Wf));
    KR_LAUNCHED();
    return KR_OK;
}
