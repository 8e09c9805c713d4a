// fused_wide.hip -- window 2^16 in one kernel: a frame's whole complex
// transform (M = 2^15 values, 256 KiB) is held in the registers of one
// workgroup.
//
// LDS (160 KiB per CU) cannot hold M complex values, but the registers of a CU
// (512 KiB) can: 1024 threads with 32 values each.  M = 32 x 32 x 32, so three
// radix-32 Stockham passes with two exchanges between them, and an exchange
// moves the real parts through LDS (128 KiB), then the imaginary parts.  A
// frame is read once and its result written once; the two passes that served
// this window before wrote and read 16 bytes of scratch per complex value in
// between.
//
// Measured, 2^27 samples, 75% overlap, Blackman, DC removal, power (8193
// frames): 1563 us in two passes (1.03 TB/s of signal and result), 810 us here
// (1.99 TB/s).  One workgroup fills a CU, so the phases of a frame follow each
// other: of 24.6 us a frame, builds without the part in question take 5.1 us
// less without the samples' loads, 3.4 with the window's from L1 instead of L2,
// 4.4 without the transforms, 3.8 without the exchanges, 4.0 without the
// stores.  A persistent grid that loads the next frame while this one's result
// goes out took 850 us (a wave's loads wait for the stores issued before them).
// Requests of few frames, which leave most CUs idle here, go through the two
// passes (run_wide in multipass.hip).
#include "buffer.hpp"
#include "engine.hpp"
#include "epilogue.hpp"
#include "stockham.hpp"
#include "twisted_dft.hpp"

namespace ostft {

namespace {

constexpr int WIDE_LOG_M = 15, WIDE_M = 1 << WIDE_LOG_M, WIDE_T = WIDE_M / 32;
constexpr int WIDE_LDS = WIDE_M + WIDE_M / 32;  // floats of the exchange: one pad per 32
static_assert(WIDE_LDS >= WIDE_M + 2, "the mirror exchange's M/2 + 1 complex values");

// One component of an exchange between radix-32 passes: value q of the thread
// goes to wr[QSTEP q], value m comes from rd[m (M/32 padded)].  The caller's
// next write to LDS follows a barrier.
template <int QSTEP>
__device__ __forceinline__ void exchange(float2 (&v)[32], float* wr, const float* rd)
{
    constexpr int RSTEP = WIDE_T + WIDE_T / 32;
    cfor<0, 32>([&](auto q) { wr[QSTEP * decltype(q)::value] = v[decltype(q)::value].x; });
    __syncthreads();
    cfor<0, 32>([&](auto m) { v[decltype(m)::value].x = rd[RSTEP * decltype(m)::value]; });
    __syncthreads();
    cfor<0, 32>([&](auto q) { wr[QSTEP * decltype(q)::value] = v[decltype(q)::value].y; });
    __syncthreads();
    cfor<0, 32>([&](auto m) { v[decltype(m)::value].y = rd[RSTEP * decltype(m)::value]; });
    __syncthreads();
}

// Pass twist w = W_M^e: w^(16 >> l) for level l
__device__ __forceinline__ void load_twist(Twist<32>& tw, const float2* __restrict__ table, uint32_t e)
{
    cfor<0, 5>([&](auto l) { tw.base[decltype(l)::value] = table[e * (16u >> decltype(l)::value)]; });
}

// One frame of a workgroup.  INSIDE: the frame lies inside the signal.
template <bool INSIDE>
__device__ __forceinline__ void wide_frame(const FusedArgs& a, const float* __restrict__ in, float* __restrict__ out,
                                           uint64_t f, float* lds, uint32_t t)
{
    constexpr int M = WIDE_M, N = 2 * M, T = WIDE_T;

    // ---- the frame's packed samples z[n] = x[2n] + i x[2n+1], n = t + T m,
    //      windowed.  All samples are in flight at once, of the window 16 values:
    //      the registers hold no more. ----
    float2 v[32];
    const uint64_t fs = f * a.hop;
    const float* const x = in + fs;
    const auto bx = buffer(x, sizeof(float) * N);
    const uint64_t left = INSIDE ? (uint64_t)N : (fs < a.L ? a.L - fs : 0);  // samples inside the signal
    auto sample = [&](uint32_t m) -> float2 {
        if constexpr (INSIDE) {
            return load2(bx, 8 * t, 8 * T * m);  // 4-byte aligned is enough
        } else {
            const uint32_t s = 2 * (t + T * m);
            return make_float2(s < left ? x[s] : 0.0f, s + 1 < left ? x[s + 1] : 0.0f);
        }
    };
    if (a.win) {
        const auto bw = buffer(a.win, sizeof(float) * N);
        float2 w[32];
        cfor<0, 16>([&](auto m) {
            constexpr int MM = decltype(m)::value;
            v[MM] = sample(MM);
            w[MM] = load2(bw, 8 * t, 8 * T * MM);
        });
        cfor<16, 32>([&](auto m) { v[decltype(m)::value] = sample(decltype(m)::value); });
        __builtin_amdgcn_sched_barrier(0);
        cfor<0, 32>([&](auto m) {
            constexpr int MM = decltype(m)::value;
            v[MM] = make_float2(v[MM].x * w[MM].x, v[MM].y * w[MM].y);
            if constexpr (MM < 16)
                w[MM + 16] = load2(bw, 8 * t, 8 * T * (MM + 16));
            if constexpr (MM % 4 == 3)
                __builtin_amdgcn_sched_barrier(0);
        });
    } else {
        cfor<0, 32>([&](auto m) { v[decltype(m)::value] = sample(decltype(m)::value); });
    }

    // ---- three radix-32 passes; value q of thread t is Z[t + T q] after the last ----
    Twist<32> tw;
    twisted_dft<32, 0, 1, false>(v, tw);
    load_twist(tw, a.tw, (t & 31u) * 32u);
    const float* const rd = lds + t + (t >> 5);
    exchange<1>(v, lds + 33 * t, rd);
    twisted_dft<32, 0, 1, true>(v, tw);
    load_twist(tw, a.tw, t);
    const float2 wt = a.tw_n[t];
    exchange<33>(v, lds + (t >> 5) * (32 * 33) + (t & 31u), rd);
    twisted_dft<32, 0, 1, true>(v, tw);

    if (a.dc && t == 0)  // subtracting the mean only moves Z[0]
        v[0] = make_float2(0.5f * (v[0].x - v[0].y), 0.5f * (v[0].y - v[0].x));

    // ---- Z[M - k] of the thread's bins k = t + T q < M/2: the upper halves
    //      through LDS, with Z[0] in the place of Z[M] ----
    float2* const zu = reinterpret_cast<float2*>(lds);  // zu[j] = Z[M/2 + j]
    cfor<16, 32>([&](auto q) { zu[t + T * (decltype(q)::value - 16)] = v[decltype(q)::value]; });
    if (t == 0)
        zu[M / 2] = v[0];
    __syncthreads();

    // ---- last radix-2 stage and output: bin k gives positions k and M + k, and
    //      by the conjugate symmetry of a real frame's spectrum M - k and N - k ----
    auto epilogue = [&](auto mode_c, auto cut_c) {
        constexpr int MODE = decltype(mode_c)::value;
        constexpr bool CUT = decltype(cut_c)::value;  // HALF_COMPLEX: the frame that out_limit cuts short
        constexpr bool HALF = MODE == OUT_POWER || MODE == OUT_HALF_SPECTRUM;
        constexpr bool CPLX = MODE == OUT_HALF_COMPLEX || MODE == OUT_HALF_SPECTRUM;
        constexpr int B = CPLX ? 8 : 4;                      // bytes of an output value
        constexpr int W = HALF ? M + 1 : N;                  // values of a frame
        const uint64_t base = f * (uint64_t)W;
        const auto bo = buffer(reinterpret_cast<char*>(out) + B * base, B * W);
        const uint64_t room = a.out_limit > base ? a.out_limit - base : 0;
        auto put = [&](uint32_t lane, uint32_t pos, float2 x2, bool conj) {  // value at position lane + pos
            if constexpr (MODE == OUT_COMPAT_POWER)
                store1(bo, B * lane, B * pos, compat_power(x2));
            else if constexpr (MODE == OUT_MAGNITUDE)
                store1(bo, B * lane, B * pos, magnitude(x2));
            else if constexpr (MODE == OUT_POWER)
                store1(bo, B * lane, B * pos, power_of(x2));
            else if (!CUT || lane + pos < room)
                store2(bo, B * lane, B * pos, conj ? conj_value_of(x2) : value_of(x2));
        };
        const float2* const zm = zu + M / 2 - t;
        const uint32_t tm = T - t;  // M - k = tm + T (31 - q)
        cfor<0, 16>([&](auto q) {
            constexpr int Q = decltype(q)::value;
            const BinPair b = finish_pair<true>(v[Q], *(zm - T * Q), cmul(wt, root<64, Q>()));
            const bool first = Q == 0 && t == 0;  // bin 0 has no mirror below N
            put(t, T * Q, b.lo, false);
            if constexpr (HALF) {
                put(tm, M - T - T * Q, b.hi, !first);
            } else {
                put(t, M + T * Q, b.hi, false);
                if (!first) {
                    put(tm, M - T - T * Q, b.hi, true);
                    put(tm, N - T - T * Q, b.lo, true);
                }
            }
        });
        if (t == 0) {  // bin M/2, its own mirror
            const BinPair b = finish_pair<true>(v[16], v[16], make_float2(0.0f, -1.0f));
            put(0, M / 2, b.lo, false);
            if constexpr (!HALF)
                put(0, M + M / 2, b.hi, false);
        }
    };
    switch (a.out_mode) {
    case OUT_COMPAT_POWER: epilogue(std::integral_constant<int, OUT_COMPAT_POWER>{}, std::false_type{}); break;
    case OUT_MAGNITUDE: epilogue(std::integral_constant<int, OUT_MAGNITUDE>{}, std::false_type{}); break;
    case OUT_HALF_COMPLEX:
        if ((f + 1) * N <= a.out_limit)
            epilogue(std::integral_constant<int, OUT_HALF_COMPLEX>{}, std::false_type{});
        else
            epilogue(std::integral_constant<int, OUT_HALF_COMPLEX>{}, std::true_type{});
        break;
    case OUT_POWER: epilogue(std::integral_constant<int, OUT_POWER>{}, std::false_type{}); break;
    case OUT_HALF_SPECTRUM: epilogue(std::integral_constant<int, OUT_HALF_SPECTRUM>{}, std::false_type{}); break;
    default: break;
    }
}

}  // namespace

__global__ void __launch_bounds__(WIDE_T) __attribute__((amdgpu_waves_per_eu(4))) stft_wide_kernel(const FusedArgs a)
{
    __shared__ __align__(16) float lds[WIDE_LDS];
    const uint64_t f = xcd_block(blockIdx.x, gridDim.x);
    const float* const in = a.in + (uint64_t)blockIdx.y * a.in_stride;
    float* const out = a.out + (uint64_t)blockIdx.y * a.out_stride;
    if (f * a.hop + 2 * WIDE_M <= a.L)
        wide_frame<true>(a, in, out, f, lds, threadIdx.x);
    else
        wide_frame<false>(a, in, out, f, lds, threadIdx.x);
}

bool wide_supported(int log_m) { return log_m == WIDE_LOG_M; }

hipError_t launch_wide(const FusedArgs& a, uint32_t count, hipStream_t s)
{
    if (a.frames == 0 || count == 0)
        return hipSuccess;
    if (a.frames > 0x7fffffffull || count > 65535u || !a.combine)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(stft_wide_kernel, dim3((uint32_t)a.frames, count), dim3(WIDE_T), 0, s, a);
    return hipGetLastError();
}

}  // namespace ostft
