// twisted_dft.hpp -- register DFTs of size 2 .. 32 with fused multiply-adds.
//
// Decimation in time: every butterfly is a +- c b with the twiddle c of its
// own level, which takes 6 fused multiply-adds (a + c b as four, a - c b =
// 2 a - (a + c b) as two) where a product and a sum and a difference take 8
// instructions.  A Stockham pass's input twiddles w^m are not multiplied in
// beforehand: with E, O the transforms of the even and odd inputs,
//     sum_m x[m] w^m W_R^(mq) = E'[q] + (w W_R^q) O'[q],
// E' and O' having twist w^2, so the twist moves into the levels' twiddles
// (level LEN uses w^(R/LEN) W_LEN^q).  A radix-32 pass with a twist is then
// 480 FMAs and 11 products by constants, against 456 instructions for the
// transform, 124 for its 31 input products and 104 to form the powers.
// Butterflies of fused multiply-adds are known from the literature on FFTs for such
// machines (E. Linzer and E. Feig, IEEE Trans. Signal Processing 41, 1993; S.
// Goedecker, SIAM J. Sci. Comput. 18, 1997); a - c b is taken as 2 a - (a + c b), which
// needs no ratio of the twiddle's parts.
#pragma once

#include "fft_device.hpp"

namespace ostft {

// cos(2 pi k / 64), k = 0 .. 16
constexpr float COS64[17] = {1.0f,
                             0.99518472667219688624f,
                             0.98078528040323044913f,
                             0.95694033573220886494f,
                             0.92387953251128675613f,
                             0.88192126434835502971f,
                             0.83146961230254523708f,
                             0.77301045336273696081f,
                             0.70710678118654752440f,
                             0.63439328416364549822f,
                             0.55557023301960222474f,
                             0.47139673682599764856f,
                             0.38268343236508977173f,
                             0.29028467725446236764f,
                             0.19509032201612826785f,
                             0.09801714032956060199f,
                             0.0f};

// W_LEN^q = exp(-2 pi i q / LEN) for q <= LEN / 4, LEN a power of two up to 64
template <int LEN, int Q>
__device__ __forceinline__ float2 root()
{
    constexpr int K = Q * (64 / LEN);
    static_assert(K >= 0 && K <= 16, "first quarter of the circle");
    return make_float2(COS64[K], -COS64[16 - K]);
}

// a, b <- a + c b, a - c b; with ROT, c stands for -i c
template <bool ROT>
__device__ __forceinline__ void butterfly(float2& a, float2& b, float2 c)
{
    const float cx = ROT ? c.y : c.x, cy = ROT ? -c.x : c.y;
    const float2 s = make_float2(fmaf(-cy, b.y, fmaf(cx, b.x, a.x)), fmaf(cy, b.x, fmaf(cx, b.y, a.y)));
    b = make_float2(fmaf(2.0f, a.x, -s.x), fmaf(2.0f, a.y, -s.y));
    a = s;
}

// the same with c = 1, or -i with ROT
template <bool ROT>
__device__ __forceinline__ void butterfly1(float2& a, float2& b)
{
    const float2 t = ROT ? make_float2(b.y, -b.x) : b;
    b = csub(a, t);
    a = cadd(a, t);
}

// The twist of a size-R transform: base[l] = w^(R >> (l + 1)), l < log2(R)
// (level LEN = 2 << l).
template <int R>
struct Twist {
    float2 base[ilog2(R)];
};

// Size-R DFT of v[OFF + STEP m], m < R, in natural order in place; with
// TWIST, input m is taken times w^m.
template <int R, int OFF, int STEP, bool TWIST, int NV>
__device__ __forceinline__ void twisted_dft(float2 (&v)[NV], const Twist<R>& tw)
{
    float2 u[R];
    cfor<0, R>([&](auto m) {
        constexpr int MM = decltype(m)::value;
        u[MM] = v[OFF + STEP * bitrev<R>(MM)];
    });
    cfor<0, ilog2(R)>([&](auto l) {
        constexpr int L = decltype(l)::value, LEN = 2 << L, HALF = LEN / 2, QUART = LEN >= 4 ? LEN / 4 : 1;
        cfor<0, QUART>([&](auto q) {
            constexpr int Q = decltype(q)::value;
            float2 c = root<LEN < 4 ? 4 : LEN, Q>();
            if constexpr (TWIST)
                c = Q == 0 ? tw.base[L] : cmul(tw.base[L], c);
            cfor<0, R, LEN>([&](auto b) {
                constexpr int B = decltype(b)::value + Q;
                if constexpr (!TWIST && Q == 0) {
                    butterfly1<false>(u[B], u[B + HALF]);
                    if constexpr (LEN >= 4)
                        butterfly1<true>(u[B + QUART], u[B + QUART + HALF]);
                } else {
                    butterfly<false>(u[B], u[B + HALF], c);
                    if constexpr (LEN >= 4)
                        butterfly<true>(u[B + QUART], u[B + QUART + HALF], c);
                }
            });
        });
    });
    cfor<0, R>([&](auto m) {
        constexpr int MM = decltype(m)::value;
        v[OFF + STEP * MM] = u[MM];
    });
}

}  // namespace ostft
