// multipass.hip -- STFT for complex transform sizes M = 2^16 .. 2^19
// (windows 2^17 .. 2^20), and 2^15 (window 2^16) where a request has few frames.
//
// Same pipeline as the fused kernel (gather + window, FFT, split epilogue),
// but the transform fits no workgroup's registers, so it is cut into two
// Stockham passes M = R0 x R1 through HBM-resident scratch (this replaces the
// EXP separate radix-2 StockHamCommon launches of OKL/EXPCommon.okl:194-245,
// one per stage, and the separate ToPower / toHalfComplexFormat passes).
//
// Both passes hold 32 complex values a thread in registers, 16384, 8192 or
// 4096 a workgroup, as R-point transforms of as many columns, and take a column in two
// register steps of fused multiply-add butterflies (twisted_dft.hpp) with one
// exchange between them, whose real and imaginary parts go through LDS in turn.
//   * first pass (R0 = 2^10 = 32 x 32): samples come from the signal (overlap
//     gather + window) straight into the registers of their butterfly, results
//     leave from the registers;
//   * last pass (R1 = 2^6 .. 2^9 = R1/16 x 16): the inter-pass twiddle is the
//     twist of its butterflies and costs no products of its own.  A block of
//     butterflies k is held together with its mirror block R0 - k (0 and R0/2
//     are their own mirrors), so both Z[k] and Z[M-k] of every output index are
//     at hand: the split epilogue (last radix-2 stage, DC correction, output
//     layout) runs there and the spectrum is written once.
// As in the fused kernel, a frame of N real samples is one complex transform
// of M = N/2 points (even samples real, odd imaginary).  DC removal is applied
// in the frequency domain: subtracting the frame mean only changes the k = 0
// terms.
//
// Bound by memory traffic (signal, scratch twice, result): with the transforms
// compiled out the passes took within 10% of their time.  Against the form before
// (16 values a thread, samples and scratch staged through LDS on their way in
// and out, 2 to 3 exchanges, VALU issue 41-72% of the time), 2^27 samples:
// window 2^18, overlap 0, default layout 594 -> 507 us, with two chunks at a time
// (below) 477 (2.15 GB moved, 4.5 TB/s; a plain copy of 2 GiB runs at 4.9); 2^20, 75%,
// power 2050 -> 1590 -> 1388 us; 2^26 samples, 75%, default layout: 2^17 853 -> 839
// -> 780, 2^18 987 -> 878 -> 821, 2^19 1040 -> 903 -> 858, 2^20 1239 -> 961 -> 908 us;
// one frame: 20-26 -> 15-20 us.
#include "../../include/occastft_hip.h"

#include <algorithm>
#include <iterator>
#include <mutex>
#include <string>

#include "batch.hpp"
#include "buffer.hpp"
#include "epilogue.hpp"
#include "multipass.hpp"
#include "stockham.hpp"
#include "twisted_dft.hpp"

namespace ostft {

hipError_t Scratch::ensure(uint64_t n)
{
    if (cap >= n)
        return hipSuccess;
    release();
    hipError_t e = hipMalloc(&a, sizeof(float2) * n);
    if (e != hipSuccess) {
        release();
        return e;
    }
    cap = n;
    return hipSuccess;
}

hipError_t Scratch::acquire(hipStream_t s)
{
    if (!done) {
        const hipError_t e = hipEventCreateWithFlags(&done, hipEventDisableTiming);
        if (e != hipSuccess) {
            done = nullptr;
            return e;
        }
    }
    return used && last != s ? hipStreamWaitEvent(s, done, 0) : hipSuccess;
}

hipError_t Scratch::handoff(hipStream_t s)
{
    const hipError_t e = hipEventRecord(done, s);
    if (e == hipSuccess) {
        last = s;
        used = true;
    }
    return e;
}

float2* Scratch::hold(const Capture& c, hipStream_t s, uint64_t n)
{
    for (const Held& h : held)
        if (h.capture == c.id && h.stream == s && h.cap >= n)
            return h.a;
    const uint64_t bytes = sizeof(float2) * n;
    if (bytes > budget || held_bytes > budget - bytes)
        return nullptr;
    Held h{c.id, s, nullptr, n};
    const AllocateInCapture allow(true);
    if (hipMalloc(&h.a, bytes) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    held.push_back(h);
    held_bytes += bytes;
    return h.a;
}

void Scratch::release()
{
    if (a && in_graph) {
        held.push_back(Held{0, nullptr, a, 0});  // for destroy(); serves no further call
        held_bytes += sizeof(float2) * cap;
    } else if (a) {
        // the last call's launches (on whatever stream) must be done with it;
        // other streams and contexts on the device are not waited for
        if (used && done)
            (void)hipEventSynchronize(done);
        (void)hipFree(a);
    }
    a = nullptr;
    cap = 0;
    in_graph = false;
}

void Scratch::destroy()
{
    release();
    for (const Held& h : held)
        (void)hipFree(h.a);
    held.clear();
    held_bytes = 0;
    if (done)
        (void)hipEventDestroy(done);
    done = nullptr;
    sides.destroy();
    used = false;
}

// The split M = R0 x R1: R0 = 2^10 = 32 x 32, R1 = 2^6 .. 2^9 = R1/16 x 16 (32 in one
// step for window 2^16)
constexpr int MP_LOG_R0 = 10, MP_R0 = 1 << MP_LOG_R0;
// Scratch of a frame is [g / 16][k][g mod 16] for butterfly g and result k of
// the first pass: a run of 16 values is a cache line and a quarter wave.
constexpr uint32_t MP_RUN = 16;

// A workgroup's threads and complex values.  512 threads: two workgroups a CU
// and longer runs in memory; 256 and 128 threads: two and four times the
// workgroups, for requests that leave CUs idle otherwise.  A frame's arithmetic
// is the same in all.
template <int THREADS>
struct Tile {
    static constexpr uint32_t ELEMS = 32 * THREADS;
    static constexpr uint32_t LDS = ELEMS + ELEMS / 32;  // floats
};

struct PassArgs {
    const float* sig;  // first pass: the signal
    uint64_t L, hop;
    uint64_t frame0, frames;  // frames [frame0, frames) of this launch; scratch row 0 = frame0
    const float* win;
    float2* dst;
    const float2* tw_r;  // W_R0^j, j < R0
};

// One component of the exchange between the two steps of R-point transforms of
// a workgroup's C columns, r1 x R2 = R: row r of column c is staged at
// r C + (r / r1) PAD + c.  Second-step butterfly g = t + T u (T threads a column
// of U butterflies each) takes rows g + r1 m, value u + U m of the thread.
template <int C, int R1STEP, int PAD, int T, int U, int COMP>
__device__ __forceinline__ void gather_step(float2 (&v)[32], const float* rd)
{
    cfor<0, 32>([&](auto i) {
        constexpr int I = decltype(i)::value, UU = I % U, MM = I / U;
        const float x = rd[T * C * UU + (R1STEP * C + PAD) * MM];
        if constexpr (COMP)
            v[I].y = x;
        else
            v[I].x = x;
    });
}

// First pass: C = 16 (8 with 256 threads, 4 with 128) butterflies g of one frame (columns),
// lanes along the columns: the samples come straight into the butterflies'
// registers and the results leave from them, in runs of C values either way.
template <int LOG_M, int THREADS>
__global__ void __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(4)))
    first_pass_kernel(const PassArgs a)
{
    constexpr uint32_t M = 1u << LOG_M, R = MP_R0, C = Tile<THREADS>::ELEMS / R, T = R / 32, STRIDE = M / R;
    constexpr uint32_t PAD = C;           // spreads the 64 / C rows 32 t of a wave over the banks
    constexpr uint32_t BPF = STRIDE / C;  // workgroups per frame
    static_assert(MP_RUN % C == 0, "a workgroup's columns share their scratch runs");
    __shared__ float lds[Tile<THREADS>::LDS];
    static_assert(Tile<THREADS>::LDS >= Tile<THREADS>::ELEMS + PAD * (R / 32), "exchange");

    const uint32_t tid = threadIdx.x, c = tid % C, t = tid / C;
    // plain workgroup order: an XCD (workgroup index mod 8) takes the same
    // columns of every frame, so its L2 holds their part of the window (2^20:
    // 512 KiB of 4 MiB); each XCD on frames of its own read it from beyond L2
    // every time, 342 against 306 us a launch of 171 frames
    const uint64_t P = a.frame0 + blockIdx.x / BPF;
    const uint32_t g0 = (blockIdx.x % BPF) * C;

    // packed samples z[n] = x[2n] + i x[2n+1], n = g + STRIDE (t + T j), windowed
    float2 v[32];
    const uint64_t fs = P * a.hop;
    const uint32_t n0 = g0 + c + STRIDE * t;
    constexpr uint32_t STEP = STRIDE * T;
    const auto bw = buffer(a.win, a.win ? 8 * M : 0);
    auto window = [&](auto sample) {
        if (a.win) {
            // of the window 16 values are in flight: the registers hold no more
            float2 w[32];
            cfor<0, 16>([&](auto j) {
                constexpr int J = decltype(j)::value;
                v[J] = sample(J);
                w[J] = load2(bw, 8 * n0, 8 * STEP * J);
            });
            cfor<16, 32>([&](auto j) { v[decltype(j)::value] = sample(decltype(j)::value); });
            __builtin_amdgcn_sched_barrier(0);
            cfor<0, 32>([&](auto j) {
                constexpr int J = decltype(j)::value;
                v[J] = make_float2(v[J].x * w[J].x, v[J].y * w[J].y);
                if constexpr (J < 16)
                    w[J + 16] = load2(bw, 8 * n0, 8 * STEP * (J + 16));
                if constexpr (J % 4 == 3)
                    __builtin_amdgcn_sched_barrier(0);
            });
        } else {
            cfor<0, 32>([&](auto j) { v[decltype(j)::value] = sample(decltype(j)::value); });
        }
    };
    if (fs + 2 * (uint64_t)(g0 + C + STRIDE * (R - 1)) <= a.L) {  // the workgroup's samples are all there
        const auto bx = buffer(a.sig + fs, 8 * M);
        window([&](uint32_t j) { return load2(bx, 8 * n0, 8 * STEP * j); });
    } else {
        const float* x = a.sig + fs;
        const uint64_t left = fs < a.L ? a.L - fs : 0;
        window([&](uint32_t j) {
            const uint32_t s = 2 * (n0 + STEP * j);
            return make_float2(s < left ? x[s] : 0.0f, s + 1 < left ? x[s + 1] : 0.0f);
        });
    }

    Twist<32> none, tw;
    twisted_dft<32, 0, 1, false>(v, none);
    // twist of the second step's butterfly t: W_R^t
    cfor<0, 5>([&](auto l) { tw.base[decltype(l)::value] = a.tw_r[t * (16u >> decltype(l)::value)]; });
    float* const wr = lds + (32 * C + PAD) * t + c;
    const float* const rd = lds + tid;
    cfor<0, 32>([&](auto q) { wr[C * decltype(q)::value] = v[decltype(q)::value].x; });
    __syncthreads();
    gather_step<C, 32, PAD, T, 1, 0>(v, rd);
    __syncthreads();
    cfor<0, 32>([&](auto q) { wr[C * decltype(q)::value] = v[decltype(q)::value].y; });
    __syncthreads();
    gather_step<C, 32, PAD, T, 1, 1>(v, rd);
    twisted_dft<32, 0, 1, true>(v, tw);

    // value i is row k = t + T i of column c
    const auto bd = buffer(a.dst + (P - a.frame0) * M + (uint64_t)(g0 / MP_RUN) * (MP_RUN * R), 8 * MP_RUN * R);
    cfor<0, 32>([&](auto i) {
        constexpr int I = decltype(i)::value;
        store2(bd, 8 * (t * MP_RUN + g0 % MP_RUN + c), 8 * T * MP_RUN * I, v[I]);
    });
}

struct LastArgs {
    const float2* src;   // first pass output
    const float2* tw_n;  // W_N^k, k < M
    // W_M^(k 2^j), k < R0: the powers the first step's twists take (2^16: the only
    // step's), side by side for the butterflies of a wave (gathered from W_N^k, they
    // would fetch as many bytes again as the scratch values)
    const float2* tw_k[9];
    const double2* tw_m;  // W_M^k, k < R0, and
    const double2* tw_r;  // W_R1^j, j < R1/16: their products are the second step's
    float* out;
    uint64_t frame0, frames, out_limit;  // frames [frame0, frames); scratch row 0 = frame0
    int32_t combine, out_mode, dc;
};

__device__ __forceinline__ double2 cmul64(double2 a, double2 b)
{
    return make_double2(fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x));
}

// Last pass: C / 2 butterflies k and their mirrors R0 - k (0 and R0/2 are their
// own) of one frame, R points each with twist W_M^k: a step of r1 = R/16 points
// and one of 16.  Loads have the lanes along a butterfly's inputs, where the
// first pass left them side by side; the exchange turns the lanes along the
// butterflies, where the output positions k + R0 q are side by side.
template <int LOG_M, int THREADS>
__global__ void __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(4)))
    last_pass_kernel(const LastArgs a)
{
    constexpr uint32_t M = 1u << LOG_M, N = 2 * M, Ns = MP_R0, R = M / Ns;
    constexpr uint32_t ELEMS = Tile<THREADS>::ELEMS, C = ELEMS / R, CB = C / 2, T = R / 32;
    constexpr uint32_t r1 = R / 16, NC = 32 / r1;  // first step: NC columns a thread,
    constexpr uint32_t CSTEP = THREADS / 16;       // so far apart
    constexpr uint32_t PAD = 4;                    // spreads the 16 rows r1 t of a wave over the banks
    constexpr uint32_t BPF = Ns / C;               // workgroups per frame
    __shared__ __align__(16) float lds[Tile<THREADS>::LDS];
    static_assert(Tile<THREADS>::LDS >= ELEMS + PAD * 16 && Tile<THREADS>::LDS >= ELEMS + 2, "exchanges");

    const uint32_t tid = threadIdx.x;
    // each XCD on frames of its own: neighbouring blocks, whose output runs
    // share cache lines, meet in one L2 (plain order: 309 against 280 us at 2^18,
    // 334 against 271 at 2^20)
    const uint32_t blk = xcd_block(blockIdx.x, gridDim.x);
    const uint64_t P = a.frame0 + blk / BPF;
    const uint32_t b = blk % BPF;
    // column c < CB: butterfly b CB + c; column CB + h: its mirror Ns - (b CB + h),
    // with Ns/2 in the place of Ns (= butterfly 0, already in column 0)
    auto butterfly = [&](uint32_t c) -> uint32_t {
        const uint32_t k = b * CB + (c & (CB - 1));
        return c < CB ? k : k == 0 ? Ns / 2 : Ns - k;
    };
    float2 v[32];
    const uint32_t c = tid % C, t = tid / C, k = butterfly(c);
    if constexpr (R == 32) {
        // one step of 32 points: scratch [g / 16][k][g mod 16], the butterfly's
        // inputs are two runs of its thread
        const auto bs = buffer(a.src + (P - a.frame0) * M, 8 * M);
        cfor<0, 16>([&](auto j) {
            constexpr uint32_t J = decltype(j)::value;
            const float4 x = load4(bs, 8 * k * MP_RUN, 8 * Ns * MP_RUN * (J / 8) + 16 * (J % 8));
            v[2 * J] = make_float2(x.x, x.y);
            v[2 * J + 1] = make_float2(x.z, x.w);
        });
        Twist<32> tw;
        cfor<0, 5>([&](auto l) { tw.base[decltype(l)::value] = a.tw_k[4 - decltype(l)::value][k]; });
        twisted_dft<32, 0, 1, true>(v, tw);
    } else {
        // inputs g = t + 16 j of butterfly k: scratch [j][k][t]; columns cg + CSTEP i
        {
            const uint32_t t = tid & 15u, cg = tid >> 4;
            const auto bs = buffer(a.src + (P - a.frame0) * M, 8 * M);
            cfor<0, NC>([&](auto i) {
                const uint32_t k = butterfly(cg + CSTEP * decltype(i)::value);
                cfor<0, r1>([&](auto j) {
                    v[decltype(i)::value * r1 + decltype(j)::value] =
                        load2(bs, 8 * (k * MP_RUN + t), 8 * Ns * MP_RUN * decltype(j)::value);
                });
            });
            float* const wr = lds + (r1 * C + PAD) * t + cg;
            cfor<0, NC>([&](auto i) {
                // twist over j: W_M^(16 k)
                constexpr int O = decltype(i)::value * r1;
                const uint32_t k = butterfly(cg + CSTEP * decltype(i)::value);
                Twist<r1> tw;
                cfor<0, ilog2(r1)>([&](auto l) {
                    tw.base[decltype(l)::value] = a.tw_k[4 + ilog2(r1) - 1 - decltype(l)::value][k];
                });
                twisted_dft<r1, O, 1, true>(v, tw);
                cfor<0, r1>([&](auto q) { wr[CSTEP * decltype(i)::value + C * decltype(q)::value] = v[O + decltype(q)::value].x; });
            });
            const float* const rd = lds + tid;
            __syncthreads();
            gather_step<C, r1, PAD, T, 2, 0>(v, rd);
            __syncthreads();
            cfor<0, NC>([&](auto i) {
                cfor<0, r1>([&](auto q) {
                    wr[CSTEP * decltype(i)::value + C * decltype(q)::value] = v[decltype(i)::value * r1 + decltype(q)::value].y;
                });
            });
            __syncthreads();
            gather_step<C, r1, PAD, T, 2, 1>(v, rd);
        }
        // second step, butterfly t + T u over 16 inputs: twist W_M^k W_R^(t + T u),
        // it and its squares formed in FP64 and rounded once (products of two float
        // tables: error 2.82 for 2.46e-7 at 2^17, power, noise; the powers read from
        // tables of M/16 entries: the same error, 2^20 719 -> 729 us, here 713)
        const double2 wk = a.tw_m[k];
        cfor<0, 2>([&](auto u) {
            constexpr int UU = decltype(u)::value;
            Twist<16> tu;
            double2 w = cmul64(wk, a.tw_r[t + T * UU]);
            cfor<0, 4>([&](auto l) {
                constexpr int L = 3 - decltype(l)::value;  // base[L] = w^(8 >> L)
                tu.base[L] = make_float2((float)w.x, (float)w.y);
                if constexpr (L > 0)
                    w = cmul64(w, w);
            });
            twisted_dft<16, UU, 2, true>(v, tu);
        });
    }
    const float2 wt = a.tw_n[k + Ns * t];
    // value i is row q = t + T i of column c: Z[k + Ns q]
    const bool k0 = b == 0 && c == 0;
    if (a.dc && k0 && t == 0)  // subtracting the mean only moves Z[0]
        v[0] = make_float2(0.5f * (v[0].x - v[0].y), 0.5f * (v[0].y - v[0].x));

    // mirrors: Z[M - (k + Ns q)] is row R - 1 - q of the mirror column (row R - q
    // of column 0 for butterfly 0, with Z[0] as its row R).  The upper rows go
    // through LDS.
    float2* const zu = reinterpret_cast<float2*>(lds);  // [row - R/2][column]
    __syncthreads();
    cfor<16, 32>([&](auto i) { zu[tid + T * C * (decltype(i)::value - 16)] = v[decltype(i)::value]; });
    if (k0 && t == 0)
        zu[ELEMS / 2] = v[0];
    __syncthreads();
    const uint32_t mc = b == 0 && (c & (CB - 1)) == 0 ? c : c ^ CB;
    const float2* const zm = zu + (R / 2 - 1 + (k0 ? 1 : 0) - t) * C + mc;

    auto epilogue = [&](auto mode_c, auto comb_c, auto cut_c) {
        constexpr int MODE = decltype(mode_c)::value;
        constexpr bool COMB = decltype(comb_c)::value;
        constexpr bool CUT = decltype(cut_c)::value;  // HALF_COMPLEX: the frame that out_limit cuts short
        constexpr bool HALF = MODE == OUT_POWER || MODE == OUT_HALF_SPECTRUM;
        static_assert(COMB || !HALF, "the layouts of N/2+1 values are of the full FFT");
        constexpr bool CPLX = MODE == OUT_HALF_COMPLEX || MODE == OUT_HALF_SPECTRUM;
        constexpr uint32_t B = CPLX ? 8 : 4;      // bytes of an output value
        constexpr uint32_t W = HALF ? M + 1 : N;  // values of a frame
        const uint64_t base = P * W;
        const auto bo = buffer(reinterpret_cast<char*>(a.out) + B * base, B * W);
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
        // bin k + Ns q gives positions k + Ns q and M further on, and by the
        // conjugate symmetry of a real frame's spectrum the mirrored two
        const uint32_t lo = k + Ns * t, hi = Ns * T - lo;  // M - (lo + Ns T i) = hi + Ns T (31 - i)
        cfor<0, 16>([&](auto i) {
            constexpr uint32_t I = decltype(i)::value, O = Ns * T * I;
            const BinPair bp = finish_pair<COMB>(v[I], *(zm - T * C * I), COMB ? cmul(wt, root<64, I>()) : wt);
            const bool first = I == 0 && k0 && t == 0;  // bin 0 has no mirror below N
            put(lo, O, bp.lo, false);
            if constexpr (HALF) {
                put(hi, M - Ns * T - O, bp.hi, !first);
            } else {
                put(lo, M + O, bp.hi, false);
                if (!first) {
                    put(hi, M - Ns * T - O, COMB ? bp.hi : bp.lo, true);
                    put(hi, N - Ns * T - O, COMB ? bp.lo : bp.hi, true);
                }
            }
        });
        if (k0 && t == 0) {  // bin M/2, its own mirror
            const BinPair bp = finish_pair<COMB>(v[16], v[16], make_float2(0.0f, -1.0f));
            put(0, M / 2, bp.lo, false);
            if constexpr (!HALF)
                put(0, M + M / 2, bp.hi, false);
        }
    };
    // one straight-line body per output layout and stage choice: the reference's
    // odd-exponent result stops before the last stage, in its own layouts
    constexpr bool VAR_COMBINE = LOG_M % 2 == 0;
    using No = std::false_type;
    using Yes = std::true_type;
    auto by_stage = [&](auto mode_c, auto cut_c) {
        if constexpr (VAR_COMBINE) {
            if (!a.combine) {
                epilogue(mode_c, No{}, cut_c);
                return;
            }
        }
        epilogue(mode_c, Yes{}, cut_c);
    };
    switch (a.out_mode) {
    case OUT_COMPAT_POWER: by_stage(std::integral_constant<int, OUT_COMPAT_POWER>{}, No{}); break;
    case OUT_MAGNITUDE: by_stage(std::integral_constant<int, OUT_MAGNITUDE>{}, No{}); break;
    case OUT_HALF_COMPLEX:
        if ((P + 1) * N <= a.out_limit)
            by_stage(std::integral_constant<int, OUT_HALF_COMPLEX>{}, No{});
        else
            by_stage(std::integral_constant<int, OUT_HALF_COMPLEX>{}, Yes{});
        break;
    case OUT_POWER: epilogue(std::integral_constant<int, OUT_POWER>{}, Yes{}, No{}); break;
    case OUT_HALF_SPECTRUM: epilogue(std::integral_constant<int, OUT_HALF_SPECTRUM>{}, Yes{}, No{}); break;
    default: break;
    }
}

namespace {

// f(integral_constant<int, LOG_M>) for a runtime log_m in 15 .. 19
template <typename F>
hipError_t with_log_m(int log_m, F&& f)
{
    switch (log_m) {
    case 15: return f(std::integral_constant<int, 15>{});
    case 16: return f(std::integral_constant<int, 16>{});
    case 17: return f(std::integral_constant<int, 17>{});
    case 18: return f(std::integral_constant<int, 18>{});
    case 19: return f(std::integral_constant<int, 19>{});
    default: return hipErrorInvalidValue;
    }
}

template <int LOG_M, int THREADS>
hipError_t launch_tiles(const PassArgs& p, const LastArgs& la, hipStream_t s)
{
    const uint64_t blocks = (p.frames - p.frame0) * ((1u << LOG_M) / Tile<THREADS>::ELEMS);
    if (blocks > 0x7fffffffull)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL((first_pass_kernel<LOG_M, THREADS>), dim3((uint32_t)blocks), dim3(THREADS), 0, s, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return e;
    hipLaunchKernelGGL((last_pass_kernel<LOG_M, THREADS>), dim3((uint32_t)blocks), dim3(THREADS), 0, s, la);
    return hipGetLastError();
}

// Requests of up to so many values take the workgroups of 256 threads.  Per
// call, 512 against 256 threads (overlap 0, default layout): window 2^17, 1 frame
// 22.7 / 18.3 us, 16 frames (1.0 M values) 27.2 / 21.5, 64 (4.2 M) 37.3 / 37.4, 128
// 68.0 / 79.0; 2^20, 4 frames (2.1 M) 31.3 / 29.1, 8 (4.2 M) 39.8 / 42.2, 16 71.7 / 95.7.
constexpr uint64_t SMALL_VALUES = (uint64_t)192 * 16384;
// Up to 160 workgroups of 128 threads leave every one a CU of its own.  256 / 128
// threads, overlap 0, power: 2^16, 5 frames 18.0 / 15.7 us, 20 (0.66 M values) 19.6 /
// 17.6, 36 20.8 / 23.2; 2^17, 2 frames 16.8 / 15.5, 10 (0.66 M) 18.7 / 18.1, 14 19.4 /
// 20.3; 2^18, 2 frames 17.3 / 16.0, 4 (0.52 M) 18.1 / 17.2, 7 19.5 / 20.5; 2^19, 2 (0.52
// M) 18.4 / 17.6, 3 19.3 / 19.4.  At 2^20 their output runs are four values: one
// frame, complex half, 19.9 / 22.8.
constexpr uint64_t TINY_VALUES = (uint64_t)160 * 4096;

hipError_t launch_passes(int log_m, const PassArgs& p, const LastArgs& la, hipStream_t s)
{
    return with_log_m(log_m, [&](auto lc) -> hipError_t {
        constexpr int LOG_M = decltype(lc)::value;
        const uint64_t values = (p.frames - p.frame0) << LOG_M;
        if constexpr (LOG_M <= 18) {
            if (values <= TINY_VALUES)
                return launch_tiles<LOG_M, 128>(p, la, s);
        }
        if constexpr (LOG_M >= 16) {
            if (values > SMALL_VALUES)
                return launch_tiles<LOG_M, 512>(p, la, s);
        }
        return launch_tiles<LOG_M, 256>(p, la, s);
    });
}

}  // namespace

bool multipass_supported(int log_m) { return log_m >= 15 && log_m <= 19; }

uint64_t multipass_chunk_frames(uint64_t budget, int log_m)
{
    const uint64_t n = budget / (sizeof(float2) << log_m);
    return n ? n : 1;
}

namespace {

// The twiddle tables of the two passes (resident in the context).  With
// `noalloc` a table that is not resident yet is an error instead of being
// built.
struct PassTables {
    const float2 *r0, *k[9] = {};
    const double2 *m = nullptr, *r = nullptr;
};

// the powers W_M^(k 2^j) that the last pass reads start with this j
int first_power(int log_m) { return log_m > 15 ? 4 : 0; }

int pass_tables(ostft_ctx* ctx, int log_m, bool noalloc, PassTables* t)
{
    int rc = OSTFT_OK;
    t->r0 = ctx_twiddles(ctx, MP_R0, MP_R0, &rc, noalloc);
    for (int j = first_power(log_m); rc == OSTFT_OK && j < log_m - MP_LOG_R0; ++j)
        t->k[j] = ctx_twiddles(ctx, (int64_t)1 << (log_m - j), MP_R0, &rc, noalloc);
    if (rc == OSTFT_OK && first_power(log_m) > 0) {
        const int64_t R1 = (int64_t)1 << (log_m - MP_LOG_R0);
        if ((t->m = ctx_twiddles64(ctx, (int64_t)1 << log_m, MP_R0, &rc, noalloc)))
            t->r = ctx_twiddles64(ctx, R1, R1 / 16, &rc, noalloc);
    }
    return rc;
}

// those of window 2^16
bool wide_tables_resident(ostft_ctx* ctx, int log_m)
{
    bool all = ctx_has_twiddles(ctx, MP_R0, MP_R0);
    for (int j = 0; all && j < log_m - MP_LOG_R0; ++j)
        all = ctx_has_twiddles(ctx, (int64_t)1 << (log_m - j), MP_R0);
    return all;
}

// Frames go through both passes a chunk at a time, so that the last pass reads
// scratch that is still in the 256 MB memory-side cache.  One chunk at a time:
// 768 workgroups (96 MiB of scratch); what is left over joins the last chunk, of 1152
// (144 MiB) at most, or makes one of at least half the size.  Requests of more than
// 2304 workgroups a pass run two chunks of 512 (one round of the GPU) at a time,
// every other one on a side stream: the last workgroups of one chunk's launch leave
// the GPU to the other chunk's, and one's loads meet the other's transforms.  The
// fork and join of the streams cost 10-20 us.  One / two at a time, calls in a row
// and each waited for: power, 75%, 2^17, 2080 workgroups 196 / 204 and 205 / 224 us,
// 2400 224 / 217 and 233 / 237, 3200 300 / 289 and 316 / 310; 2^20, 2080 209 / 206 and
// 218 / 225, 2500 242 / 233 and 252 / 252, 4096 396 / 365 and 413 / 387; default layout,
// overlap 0, 2^17, 2200 250 / 253 and 260 / 272, 2500 285 / 269 and 294 / 288.  Scratch of one
// chunk at a time of 64 / 96 / 128 / 256 / 1024 MiB, 2^26 samples, 75%, default
// layout: 2^17 894 / 848 / 866 / 997 / 892 us; two at a time of 48 / 64 / 80 / 96 MiB each:
// 805 / 773 / 863 / 890.
struct Chunks {
    uint64_t want;  // frames
    bool two;       // two at a time
};
Chunks chunks_of(uint64_t frames, uint64_t room, int log_m, int out_mode)
{
    const uint64_t values = frames << log_m, tile = 16384;
    // the complex layout writes 16 bytes a value, which at 2^19 and 2^20 push the
    // second chunk's scratch out of the cache: 577 / 600 and 625 / 673 us (2^18 589 / 576)
    const bool wide = out_mode == OUT_HALF_COMPLEX && log_m >= 18;
    // and the layouts of 8 bytes a value at 2^20 gain from twice as many workgroups on:
    // default, overlap 0.5, 2300 273 / 278, 4096 486 / 465; 75%, 2300 262 / 269, 2800
    // 319 / 322, 4096 473 / 462; overlap 0, 2300 288 / 299, 4096 517 / 521, 8192 1023 / 1018
    const uint64_t from = log_m == 19 && out_mode != OUT_POWER ? 4096 : 2304;
    Chunks c;
    c.two = values > from * tile && room >= 2 * ((512 * tile) >> log_m) && !wide;
    c.want = ((c.two ? 512 : 768) * tile) >> log_m;
    return c;
}
// the most frames of one chunk
uint64_t chunk_most(const Chunks& c, uint64_t frames) { return std::min(c.two ? c.want : c.want + c.want / 2, frames); }
// frames of the next chunk with `left` to go and scratch for `cap`
uint64_t chunk_frames(const Chunks& c, uint64_t left, uint64_t cap)
{
    if (cap < std::min(chunk_most(c, left), left)) {  // a small budget: equal chunks
        const uint64_t n = (left + cap - 1) / cap;
        return (left + n - 1) / n;
    }
    if (c.two)
        return left <= c.want ? left : left < 2 * c.want ? (left + 1) / 2 : c.want;
    return left <= c.want + c.want / 2 ? left : c.want;
}

// Both passes over the request's frames, chunk by chunk through `buf` (`cap`
// frames; two such buffers with `other`, which takes every other chunk).
int run_chunks(ostft_ctx* ctx, int log_m, const FusedArgs& a, const PassTables& t, float2* buf, uint64_t cap,
               const Chunks& c, hipStream_t s, SideStream* other = nullptr)
{
    PassArgs p;
    p.sig = a.in;
    p.L = a.L;
    p.hop = a.hop;
    p.win = a.win;
    p.tw_r = t.r0;

    LastArgs la;
    la.tw_m = t.m;
    la.tw_r = t.r;
    la.tw_n = a.tw_n;
    std::copy(std::begin(t.k), std::end(t.k), la.tw_k);
    la.out = a.out;
    la.out_limit = a.out_limit;
    la.combine = a.combine;
    la.out_mode = a.out_mode;
    la.dc = a.dc;

    hipError_t e = other ? other->fork(s) : hipSuccess;
    if (e != hipSuccess)
        return ctx_hip_fail(ctx, e, "multi-pass side stream");
    uint32_t i = 0;
    for (uint64_t f0 = 0; e == hipSuccess && f0 < a.frames; f0 = p.frames, ++i) {
        const bool side = other && (i & 1u);
        p.dst = buf + (side ? cap << log_m : 0);
        la.src = p.dst;
        p.frame0 = la.frame0 = f0;
        p.frames = la.frames = f0 + chunk_frames(c, a.frames - f0, cap);
        e = launch_passes(log_m, p, la, side ? other->stream : s);
    }
    if (other) {  // also after a failed launch: what follows on s comes after the side stream's work
        const hipError_t j = other->join(s);
        e = e == hipSuccess ? j : e;
    }
    return e == hipSuccess ? OSTFT_OK : ctx_hip_fail(ctx, e, "multi-pass launch");
}

// Scratch of the allocation-free entry point: a fixed device array, one
// per GPU, shared by every such call on that GPU (calls that overlap in
// time on one GPU race on it).  Host code reaches it only through the
// address hipGetSymbolAddress returns for the device (the array's name is a
// host-side stand-in, not a device address).
constexpr uint64_t STATIC_SCRATCH_BYTES = 64ull << 20;
__device__ __align__(256) float2 scratch[STATIC_SCRATCH_BYTES / sizeof(float2)];

constexpr int MAX_DEVICES = 64;
std::mutex static_mu;
float2* static_ptr[MAX_DEVICES] = {};

}  // namespace

hipError_t multipass_static_scratch_init(int device)
{
    if (device < 0 || device >= MAX_DEVICES)
        return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(static_mu);
    if (static_ptr[device])
        return hipSuccess;
    // the caller made `device` current: this is that device's copy
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess)
        return e;
    static_ptr[device] = static_cast<float2*>(ptr);
    return hipSuccess;
}

// Window 2^16: the one kernel keeps a CU busy with a frame, so a request of few
// frames leaves the GPU idle; up to 56 frames (64 of the complex layout, whose
// stores take the one kernel longer) take the two passes, four or eight
// workgroups a frame, with the same arithmetic (M = 32 x 32 x 32 either way).  One
// kernel / two passes, power: 5 frames 23.5 / 15.7 us, 20 23.5 / 17.6, 36 23.8 / 20.8,
// 52 24.1 / 23.1, 64 24.2 / 24.8, 80 24.3 / 29.8; complex half: 3 frames 28.6 / 15.8, 48
// 28.5 / 24.7, 64 29.0 / 26.5, 96 29.0 / 32.5.
constexpr uint64_t WIDE_IN_PASSES = 56, WIDE_IN_PASSES_COMPLEX = 64;

static bool wide_in_passes(const FusedArgs& a)
{
    return a.frames <= (a.out_mode == OUT_HALF_COMPLEX ? WIDE_IN_PASSES_COMPLEX : WIDE_IN_PASSES);
}

static int run_one_kernel(ostft_ctx* ctx, const FusedArgs& a, hipStream_t s)
{
    const hipError_t e = launch_wide(a, 1, s);
    return e == hipSuccess ? OSTFT_OK : ctx_hip_fail(ctx, e, "wide STFT launch");
}

int run_wide(ostft_ctx* ctx, int log_m, const FusedArgs& a, hipStream_t s)
{
    if (wide_in_passes(a)) {
        const Capture capture = capture_of(s);
        bool room;
        {  // in chunks of a small budget the passes would be the slower form
            std::lock_guard<std::mutex> lk(ctx_scratch_mutex(ctx));
            Scratch& sc = ctx_scratch(ctx);
            room = multipass_chunk_frames(sc.budget, log_m) >= a.frames;
            // a captured call takes the passes with a buffer of its own, and tables
            // that are there (none can be built under capture)
            if (room && capture.on)
                room = wide_tables_resident(ctx, log_m) && sc.hold(capture, s, a.frames << log_m);
        }
        if (room)
            return run_multipass(ctx, log_m, a, s);
    }
    return run_one_kernel(ctx, a, s);
}

// On the context's scratch with its event, not on the fixed array: calls of this
// window may overlap in time.  One kernel / passes, power: 5 frames 23.5 / 15.5 us,
// 20 23.5 / 17.4, 40 23.8 / 20.4.
int run_wide_noalloc(ostft_ctx* ctx, int log_m, const FusedArgs& a, hipStream_t s)
{
    if (wide_in_passes(a) && wide_tables_resident(ctx, log_m)) {
        const int rc = run_multipass(ctx, log_m, a, s, true);
        if (rc != OSTFT_ERR_NOT_PREPARED)
            return rc;
    }
    return run_one_kernel(ctx, a, s);
}

int run_multipass(ostft_ctx* ctx, int log_m, const FusedArgs& a, hipStream_t s, bool noalloc)
{
    if (!multipass_supported(log_m))
        return OSTFT_ERR_UNSUPPORTED;
    const uint64_t M = 1ull << log_m;
    // one call at a time queues launches on the shared scratch; the event
    // chain (acquire / handoff) orders their GPU work across streams
    std::lock_guard<std::mutex> lk(ctx_scratch_mutex(ctx));
    Scratch& sc = ctx_scratch(ctx);
    const uint64_t room = multipass_chunk_frames(sc.budget, log_m);
    const Chunks c = chunks_of(a.frames, room, log_m, a.out_mode);
    const uint64_t cap = std::min(room, chunk_most(c, a.frames));
    const uint64_t need = (c.two ? 2 : 1) * cap * M;
    const Capture capture = capture_of(s);
    if (noalloc && (capture.on || cap < a.frames || sc.cap < need))
        return OSTFT_ERR_NOT_PREPARED;
    float2* buf = capture.on ? sc.hold(capture, s, need) : nullptr;
    hipError_t e = hipSuccess;
    if (!buf) {
        const AllocateInCapture allow(capture.on);
        e = sc.ensure(need);
        if (e != hipSuccess)
            return ctx_hip_fail(ctx, e, "multi-pass scratch allocation");
        buf = sc.a;
        sc.in_graph |= capture.on;
    }
    if (!capture.on)  // a graph's launches are ordered by who replays it
        e = sc.acquire(s);
    if (e != hipSuccess)
        return ctx_hip_fail(ctx, e, "multi-pass scratch ordering");
    PassTables t;
    int rc = pass_tables(ctx, log_m, false, &t);
    if (rc == OSTFT_OK)
        rc = run_chunks(ctx, log_m, a, t, buf, cap, c, s, c.two ? &sc.sides.of(capture) : nullptr);
    // also after a failed launch: what was queued may still use the scratch
    if (!capture.on)
        e = sc.handoff(s);
    if (rc != OSTFT_OK)
        return rc;
    return e == hipSuccess ? OSTFT_OK : ctx_hip_fail(ctx, e, "multi-pass scratch event");
}

int run_multipass_static(ostft_ctx* ctx, int device, int log_m, const FusedArgs& a, hipStream_t s)
{
    if (!multipass_supported(log_m))
        return OSTFT_ERR_UNSUPPORTED;
    const uint64_t frame_bytes = sizeof(float2) << log_m;
    if (frame_bytes > STATIC_SCRATCH_BYTES)
        return ctx_fail(ctx, OSTFT_ERR_TOO_LARGE,
                        "one frame's intermediate spectrum (" + std::to_string(frame_bytes)
                            + " B) exceeds the fixed scratch of the allocation-free entry point ("
                            + std::to_string(STATIC_SCRATCH_BYTES) + " B)");
    float2* buf = nullptr;
    {
        std::lock_guard<std::mutex> lk(static_mu);
        buf = device >= 0 && device < MAX_DEVICES ? static_ptr[device] : nullptr;
    }
    if (!buf)
        return ctx_fail(ctx, OSTFT_ERR_HIP, "fixed scratch of this device was not set up at context creation");
    PassTables t;
    const int rc = pass_tables(ctx, log_m, true, &t);
    if (rc != OSTFT_OK)
        return rc;
    Chunks c = chunks_of(a.frames, 0, log_m, a.out_mode);  // no other stream, no event
    return run_chunks(ctx, log_m, a, t, buf, std::min(STATIC_SCRATCH_BYTES / frame_bytes, a.frames), c, s);
}

}  // namespace ostft
