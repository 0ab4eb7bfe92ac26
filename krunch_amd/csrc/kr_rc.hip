// Range-coder kernels and their C-ABI entry points.
//
// The coder is serial within a stream. Runs of symbols (kr_encode_step,
// kr_encode_pairs_batched) are encoded by one wave per stream, the lockstep
// calls of one symbol per stream by one lane per stream. The entry points keep
// the reference's argument meaning and state layout (krunch_ac/cuda/main.cpp
// encode_step / decode_step and their _batched forms; encode_kernel.cu,
// decode_kernel.cu) and add buffer bounds: output writes stop at out_cap, input
// reads past a stream's limit return zeros.
#include "kr_rc_device.h"

namespace {

constexpr int kRcThreads = 64;

__device__ __forceinline__ uint32_t stream_base(const int32_t* base, int b) {
    return base ? (uint32_t)base[b] : 0u;
}

__device__ __forceinline__ void note_overflow(uint32_t* err, uint32_t overflow) {
    if (overflow && err) atomicOr(err, 1u);
}

// Symbols outside [0, V) would index past a CDF row: clamp and flag (bit 1).
__device__ __forceinline__ int checked_symbol(int s, int V, uint32_t* err) {
    if (s < 0 || s >= V) {
        if (err) atomicOr(err, 2u);
        return 0;
    }
    return s;
}

// ---------------------------------------------------------------------------
// Encoding a run of symbols with one wave per stream.
//
// The state recursion (narrow, shift out shared bits, E3) is serial, but the
// bits it emits are not needed by it. So per batch of 64 symbols the wave
// loads one interval per lane, runs the recursion as scalar code (an
// interval read by v_readlane, ~30 scalar instructions per symbol; the spec's
// two renormalisations in the closed form of kr_rc_encode) and leaves each
// symbol's shift counts and interval bottom in lane i. The lanes then place
// their symbols' bits in parallel: a scan over the E3 counts gives the
// complements each emission carries, a scan over the lengths its position,
// and the bits are OR-ed into an LDS window that leaves as whole words.
// Bound: the latency of the scalar chain. One lane per stream doing all of it
// (a memory round trip, ~60 dependent vector instructions and the bit writer
// per symbol) took 388 us for 1000 symbols and 0.76 ms for 256 streams x 1024 on
// MI355X; this takes 116 us for the latter.
// ---------------------------------------------------------------------------
constexpr int kWinWords = 136;                 // bit window of a batch
// A batch emits at most 64 x (32 shared bits + 30 E3 bits) plus the
// complements carried in; with more than this carried in, lane 0 writes the
// batch's bits serially instead.
constexpr uint32_t kWinPending = 256;
static_assert(64 * 62 + kWinPending + 32 <= 32 * kWinWords, "a batch's bits fit the window");

__device__ __forceinline__ int wave_incl_sum(int v, int lane) {
    #pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int up = __shfl_up(v, o);
        if (lane >= o) v += up;
    }
    return v;
}

// OR the n low bits of v (1 <= n <= 32) into the window at bit position pos.
__device__ __forceinline__ void window_or(uint32_t* win, uint32_t pos, uint32_t v, uint32_t n) {
    const uint32_t a = v << (32u - n), off = pos & 31u;
    atomicOr(&win[pos >> 5], a >> off);
    if (off + n > 32u) atomicOr(&win[(pos >> 5) + 1], a << (32u - off));
}

// Symbols i = 0 .. n - 1 with intervals fetch(i) -> uint2 (cdf[sym],
// cdf[sym + 1]) onto the stream at out, whole wave. Same bytes and state as n
// calls of kr_rc_encode. Returns whether a byte at or past cap was dropped.
template <class Fetch>
__device__ __forceinline__ uint32_t encode_run(Fetch fetch, int n, uint8_t* out, uint32_t cap,
                                               kr_rc_state& st, int prec, uint32_t* win, int lane) {
    uint32_t low = __builtin_amdgcn_readfirstlane(st.low);
    uint32_t hb = __builtin_amdgcn_readfirstlane(~st.high);      // the complement of high
    uint32_t pending = __builtin_amdgcn_readfirstlane(st.pending_or_value);
    const uint32_t bit0 = __builtin_amdgcn_readfirstlane(st.bit_offset);
    uint32_t byte = bit0 >> 3;                  // first byte of the window
    uint32_t nacc = bit0 & 7u;                  // bits of it already there
    uint32_t overflow = 0;
    for (int w = lane; w < kWinWords; w += 64) win[w] = 0;
    __builtin_amdgcn_wave_barrier();
    if (nacc && lane == 0)
        win[0] = ((byte < cap ? (uint32_t)out[byte] : 0u) & ((0xFF00u >> nacc) & 0xFFu)) << 24;
    __builtin_amdgcn_wave_barrier();

    uint2 next = fetch(min(lane, n - 1));
    for (int i0 = 0; i0 < n; i0 += 64) {
        const uint2 iv = next;
        const int cnt = min(64, n - i0);
        if (i0 + 64 < n) next = fetch(min(i0 + 64 + lane, n - 1));
        // ---- the recursion: symbol i's record into lane i
        int rec = 0, rlow = 0;                  // n1 | k << 8, and low after narrowing
        for (int i = 0; i < cnt; i++) {
            const uint32_t c_lo = __builtin_amdgcn_readlane(iv.x, i);
            const uint32_t c_hi = __builtin_amdgcn_readlane(iv.y, i);
            const uint32_t d = ~hb - low;       // span - 1
            const uint32_t x = (uint32_t)(((uint64_t)d * c_lo + c_lo) >> prec);
            const uint32_t y = (uint32_t)(((uint64_t)d * c_hi + c_hi) >> prec);
            hb = 0u - (low + y);                // ~(low + y - 1)
            low = low + x;
            const uint32_t n1 = __clz(~(low ^ hb));
            const bool mine = lane == i;
            rlow = mine ? (int)low : rlow;
            low <<= n1;
            hb <<= n1;
            // low = 0..., high = 1...: k E3 steps keep the top bits as they are
            uint32_t k = __clz(~(low & hb) << 1);
            k = k > 30u ? 30u : k;
            rec = mine ? (int)(n1 | (k << 8)) : rec;
            low = (low << k) & 0x7FFFFFFFu;
            hb = (hb << k) & 0x7FFFFFFFu;
        }
        // ---- the bits: lane i places symbol i's
        const uint32_t n1 = lane < cnt ? (uint32_t)rec & 0xFFu : 0u;
        const uint32_t k = lane < cnt ? (uint32_t)rec >> 8 : 0u;
        const bool emits = n1 != 0;
        // complements carried: E3 steps since the last emission before this lane
        const int ksum = wave_incl_sum((int)k, lane);
        const unsigned long long em = __ballot(emits);
        const unsigned long long below = em & ((1ull << lane) - 1ull);
        const int last = below ? 63 - __clzll(below) : -1;
        const int kbefore = __shfl(ksum - (int)k, last < 0 ? 0 : last);   // E3 sum before symbol `last`
        const uint32_t pend = (uint32_t)(ksum - (int)k - (last < 0 ? 0 : kbefore)) +
                              (last < 0 ? pending : 0u);
        const uint32_t len = emits ? n1 + pend : 0u;
        const uint32_t carried = pending;       // into the batch's first emission
        const int le = em ? 63 - __clzll(em) : -1;
        const int ktot = __builtin_amdgcn_readlane(ksum, 63);
        pending = le < 0 ? pending + (uint32_t)ktot
                         : (uint32_t)(ktot - __builtin_amdgcn_readlane(ksum - (int)k, le));
        const uint32_t b0 = (uint32_t)rlow >> 31;
        if (carried <= kWinPending) {
            const int incl = wave_incl_sum((int)len, lane);
            const uint32_t total = nacc + (uint32_t)__builtin_amdgcn_readlane(incl, 63);
            if (emits) {
                uint32_t pos = nacc + (uint32_t)incl - len;
                window_or(win, pos, b0, 1u);
                pos++;
                if (b0) pos += pend;            // complements are zeros
                else
                    for (uint32_t left = pend; left; ) {
                        const uint32_t m = left < 32u ? left : 32u;
                        window_or(win, pos, 0xFFFFFFFFu >> (32u - m), m);
                        pos += m;
                        left -= m;
                    }
                if (n1 > 1u)
                    window_or(win, pos, ((uint32_t)rlow >> (32u - n1)) & ((1u << (n1 - 1u)) - 1u), n1 - 1u);
            }
            __builtin_amdgcn_wave_barrier();
            // whole words leave, the rest moves to the front
            const uint32_t nw = total >> 5;
            for (uint32_t w = lane; w < nw; w += 64) {
                const uint32_t v = win[w];
                #pragma unroll
                for (uint32_t e = 0; e < 4u; e++) {
                    const uint32_t idx = byte + 4u * w + e;
                    if (idx < cap) out[idx] = (uint8_t)(v >> (24u - 8u * e));
                    else overflow = 1;
                }
            }
            const uint32_t rest = win[nw];
            __builtin_amdgcn_wave_barrier();
            for (uint32_t w = lane; w <= nw; w += 64) win[w] = w == 0 ? rest : 0u;
            __builtin_amdgcn_wave_barrier();
            byte += 4u * nw;
            nacc = total & 31u;
        } else {
            // (never in practice) a long run of complements: lane 0 writes the
            // batch's bits one symbol at a time
            kr_bit_sink sink;
            sink.buf = out;
            sink.byte = byte;
            sink.acc = (uint64_t)win[0] << 32;
            sink.nacc = nacc;
            sink.cap = cap;
            sink.overflow = 0;
            for (int i = 0; i < cnt; i++) {
                const uint32_t e1 = __builtin_amdgcn_readlane(n1, i), ep = __builtin_amdgcn_readlane(pend, i);
                const uint32_t el = __builtin_amdgcn_readlane(rlow, i);
                if (e1 == 0 || lane != 0) continue;
                sink.put_bits(el >> 31, 1u);
                sink.put_run((el >> 31) ^ 1u, ep);
                if (e1 > 1u) sink.put_bits((el >> (32u - e1)) & ((1u << (e1 - 1u)) - 1u), e1 - 1u);
            }
            overflow |= sink.overflow;
            byte = __builtin_amdgcn_readfirstlane(sink.byte);
            nacc = __builtin_amdgcn_readfirstlane(sink.nacc);
            if (lane == 0) win[0] = (uint32_t)(sink.acc >> 32);
            __builtin_amdgcn_wave_barrier();
        }
    }
    // the remaining bits: whole bytes and the last, partial one
    const uint32_t v = win[0];
    for (uint32_t e = lane; 8u * e < nacc; e += 64) {
        if (byte + e < cap) out[byte + e] = (uint8_t)(v >> (24u - 8u * e));
        else overflow = 1;
    }
    st.low = low;
    st.high = ~hb;
    st.pending_or_value = pending;
    st.bit_offset = byte * 8u + nacc;
    return overflow;
}

// N rows of one stream, full CDF rows (cdf_stride entries per row); one wave.
__global__ void __launch_bounds__(64)
rc_encode_rows_kernel(const int32_t* __restrict__ cdf, int cdf_stride,
                      const int32_t* __restrict__ symbols, int N, uint8_t* out, uint32_t out_cap,
                      kr_rc_state* state, int prec, uint32_t* err) {
    __shared__ uint32_t win[kWinWords];
    const int lane = threadIdx.x;
    kr_rc_state st = *state;
    auto fetch = [&](int i) {
        const int32_t* row = cdf + (size_t)i * (size_t)cdf_stride;
        const int s = checked_symbol(symbols[i], cdf_stride - 1, err);
        return make_uint2((uint32_t)row[s], (uint32_t)row[s + 1]);
    };
    const uint32_t overflow = encode_run(fetch, N, out, out_cap, st, prec, win, lane);
    if (lane == 0) *state = st;
    note_overflow(err, overflow);
}

// One symbol per stream, CDF rows [B, V+1].
__global__ void rc_encode_step_batched_kernel(const int32_t* __restrict__ cdfs, int V,
                                              const int32_t* __restrict__ symbols,
                                              uint8_t* __restrict__ out, uint32_t out_cap,
                                              const int32_t* __restrict__ base,
                                              kr_rc_state* states, int B, int prec,
                                              uint32_t* err) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B) return;
    const uint32_t o = stream_base(base, b);
    const int32_t* row = cdfs + (size_t)b * (size_t)(V + 1);
    kr_rc_state st = states[b];
    kr_bit_sink sink;
    sink.open(out + o, st.bit_offset, out_cap > o ? out_cap - o : 0u);
    const int s = checked_symbol(symbols[b], V, err);
    kr_rc_encode(st.low, st.high, st.pending_or_value, (uint32_t)row[s], (uint32_t)row[s + 1],
                 prec, sink);
    st.bit_offset = sink.close();
    states[b] = st;
    note_overflow(err, sink.overflow);
}

// T symbols per stream from precomputed intervals: pairs[b*pair_stride + t] =
// (cdf[sym], cdf[sym+1]). Equivalent to T calls of the batched step. One wave
// per stream.
__global__ void __launch_bounds__(64)
rc_encode_pairs_kernel(const uint2* __restrict__ pairs, int T, long long pair_stride,
                       const int32_t* __restrict__ n_valid, uint8_t* out, uint32_t out_cap,
                       const int32_t* __restrict__ base, kr_rc_state* states, int prec,
                       uint32_t* err) {
    __shared__ uint32_t win[kWinWords];
    const int b = blockIdx.x, lane = threadIdx.x;
    int n = T;
    if (n_valid) n = max(0, min(T, (int)n_valid[b]));
    n = __builtin_amdgcn_readfirstlane(n);
    if (n == 0) return;
    const uint32_t o = stream_base(base, b);
    kr_rc_state st = states[b];
    const uint2* p = pairs + (size_t)b * (size_t)pair_stride;
    const uint32_t overflow = encode_run([&](int i) { return p[i]; }, n, out + o,
                                         out_cap > o ? out_cap - o : 0u, st, prec, win, lane);
    if (lane == 0) states[b] = st;
    note_overflow(err, overflow);
}

__global__ void rc_encode_finalize_kernel(uint8_t* __restrict__ out, uint32_t out_cap,
                                          const int32_t* __restrict__ base, kr_rc_state* states,
                                          int B, uint32_t* err) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B) return;
    const uint32_t o = stream_base(base, b);
    kr_rc_state st = states[b];
    kr_bit_sink sink;
    sink.open(out + o, st.bit_offset, out_cap > o ? out_cap - o : 0u);
    kr_rc_flush(st.low, st.pending_or_value, sink);
    st.bit_offset = sink.close();
    st.pending_or_value = 0;
    states[b] = st;
    note_overflow(err, sink.overflow);
}

__device__ __forceinline__ kr_bit_source open_source(const uint8_t* in, uint32_t in_len,
                                                     const int32_t* base, const int32_t* limits,
                                                     int b, uint32_t bitpos) {
    kr_bit_source src;
    const uint32_t o = stream_base(base, b);
    uint32_t lim = in_len > o ? in_len - o : 0u;
    if (limits && (uint32_t)limits[b] < lim) lim = (uint32_t)limits[b];
    src.buf = in + (o < in_len ? o : 0u);
    src.limit = lim;
    src.pos = bitpos;
    return src;
}

__global__ void rc_decode_init_kernel(const uint8_t* __restrict__ in, uint32_t in_len,
                                      const int32_t* __restrict__ base,
                                      const int32_t* __restrict__ limits, kr_rc_state* states,
                                      int B) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B) return;
    kr_bit_source src = open_source(in, in_len, base, limits, b, 0u);
    uint32_t value = 0;
    for (int i = 0; i < 32; i++) value = (value << 1) | src.get();
    kr_rc_state st;
    st.low = 0;
    st.high = 0xFFFFFFFFu;
    st.pending_or_value = value;
    st.bit_offset = src.pos;
    states[b] = st;
}

__global__ void rc_decode_step_kernel(const int32_t* __restrict__ cdfs, int V,
                                      const uint8_t* __restrict__ in, uint32_t in_len,
                                      const int32_t* __restrict__ base,
                                      const int32_t* __restrict__ limits, kr_rc_state* states,
                                      int32_t* __restrict__ out_syms, int B, int prec) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B) return;
    const int32_t* row = cdfs + (size_t)b * (size_t)(V + 1);
    kr_rc_state st = states[b];
    kr_bit_source src = open_source(in, in_len, base, limits, b, st.bit_offset);
    const uint32_t target = kr_rc_target(st.low, st.high, st.pending_or_value, prec);
    int lo = 0, hi = V;                 // largest sym with cdf[sym] <= target
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if ((uint32_t)row[mid + 1] <= target) lo = mid + 1;
        else hi = mid;
    }
    const int sym = lo < V ? lo : V - 1;
    out_syms[b] = sym;
    kr_rc_consume(st.low, st.high, st.pending_or_value, (uint32_t)row[sym],
                  (uint32_t)row[sym + 1], prec, src);
    st.bit_offset = src.pos;
    states[b] = st;
}

inline int blocks_for(int B) { return (B + kRcThreads - 1) / kRcThreads; }

}  // namespace

extern "C" {

int kr_encode_step(const int32_t* cdf, int cdf_stride, const int32_t* symbols, int N,
                   uint8_t* output_buf, uint32_t out_cap, uint32_t* state, int cdf_precision,
                   uint32_t* err_flag, void* stream) {
    KR_REQUIRE(cdf && symbols && output_buf && state, "kr_encode_step: null pointer");
    KR_REQUIRE(N >= 0 && cdf_stride >= 2, "kr_encode_step: bad N=%d or stride=%d", N, cdf_stride);
    KR_REQUIRE(cdf_precision >= 1 && cdf_precision <= 31, "bad cdf_precision %d", cdf_precision);
    if (N == 0) return KR_OK;
    rc_encode_rows_kernel<<<1, 64, 0, kr_stream(stream)>>>(
        cdf, cdf_stride, symbols, N, output_buf, out_cap, reinterpret_cast<kr_rc_state*>(state),
        cdf_precision, err_flag);
    KR_LAUNCHED();
    return KR_OK;
}

int kr_encode_finalize(uint8_t* output_buf, uint32_t out_cap, uint32_t* state,
                       uint32_t* err_flag, void* stream) {
    KR_REQUIRE(output_buf && state, "kr_encode_finalize: null pointer");
    rc_encode_finalize_kernel<<<1, kRcThreads, 0, kr_stream(stream)>>>(
        output_buf, out_cap, nullptr, reinterpret_cast<kr_rc_state*>(state), 1, err_flag);
    KR_LAUNCHED();
    return KR_OK;
}

int kr_encode_step_batched(const int32_t* cdfs, int V, const int32_t* symbols,
                           uint8_t* output_buf, uint32_t out_cap,
                           const int32_t* base_byte_offsets, uint32_t* states, int B,
                           int cdf_precision, uint32_t* err_flag, void* stream) {
    KR_REQUIRE(cdfs && symbols && output_buf && base_byte_offsets && states,
               "kr_encode_step_batched: null pointer");
    KR_REQUIRE(V >= 1 && B >= 0, "kr_encode_step_batched: bad V=%d B=%d", V, B);
    if (B == 0) return KR_OK;
    rc_encode_step_batched_kernel<<<blocks_for(B), kRcThreads, 0, kr_stream(stream)>>>(
        cdfs, V, symbols, output_buf, out_cap, base_byte_offsets,
        reinterpret_cast<kr_rc_state*>(states), B, cdf_precision, err_flag);
    KR_LAUNCHED();
    return KR_OK;
}

int kr_encode_pairs_batched(const uint32_t* pairs, int T, long long pair_stride,
                            const int32_t* n_valid, uint8_t* output_buf, uint32_t out_cap,
                            const int32_t* base_byte_offsets, uint32_t* states, int B,
                            int cdf_precision, uint32_t* err_flag, void* stream) {
    KR_REQUIRE(pairs && output_buf && states, "kr_encode_pairs_batched: null pointer");
    KR_REQUIRE(T >= 0 && B >= 0 && pair_stride >= T, "kr_encode_pairs_batched: bad shape");
    if (B == 0 || T == 0) return KR_OK;
    rc_encode_pairs_kernel<<<B, 64, 0, kr_stream(stream)>>>(
        reinterpret_cast<const uint2*>(pairs), T, pair_stride, n_valid, output_buf, out_cap,
        base_byte_offsets, reinterpret_cast<kr_rc_state*>(states), cdf_precision, err_flag);
    KR_LAUNCHED();
    return KR_OK;
}

int kr_encode_finalize_batched(uint8_t* output_buf, uint32_t out_cap,
                               const int32_t* base_byte_offsets, uint32_t* states, int B,
                               uint32_t* err_flag, void* stream) {
    KR_REQUIRE(output_buf && states, "kr_encode_finalize_batched: null pointer");
    if (B == 0) return KR_OK;
    rc_encode_finalize_kernel<<<blocks_for(B), kRcThreads, 0, kr_stream(stream)>>>(
        output_buf, out_cap, base_byte_offsets, reinterpret_cast<kr_rc_state*>(states), B,
        err_flag);
    KR_LAUNCHED();
    return KR_OK;
}

int kr_decode_init_batched(const uint8_t* input_buf, uint32_t in_len,
                           const int32_t* base_byte_offsets, const int32_t* byte_limits,
                           uint32_t* states, int B, void* stream) {
    KR_REQUIRE(input_buf && states, "kr_decode_init_batched: null pointer");
    if (B == 0) return KR_OK;
    rc_decode_init_kernel<<<blocks_for(B), kRcThreads, 0, kr_stream(stream)>>>(
        input_buf, in_len, base_byte_offsets, byte_limits, reinterpret_cast<kr_rc_state*>(states),
        B);
    KR_LAUNCHED();
    return KR_OK;
}

int kr_decode_step_batched(const int32_t* cdfs, int V, const uint8_t* input_buf, uint32_t in_len,
                           const int32_t* base_byte_offsets, const int32_t* byte_limits,
                           uint32_t* states, int32_t* out_syms, int B, int cdf_precision,
                           void* stream) {
    KR_REQUIRE(cdfs && input_buf && states && out_syms, "kr_decode_step_batched: null pointer");
    KR_REQUIRE(V >= 1, "kr_decode_step_batched: bad V=%d", V);
    if (B == 0) return KR_OK;
    rc_decode_step_kernel<<<blocks_for(B), kRcThreads, 0, kr_stream(stream)>>>(
        cdfs, V, input_buf, in_len, base_byte_offsets, byte_limits,
        reinterpret_cast<kr_rc_state*>(states), out_syms, B, cdf_precision);
    KR_LAUNCHED();
    return KR_OK;
}

}  // extern "C"
