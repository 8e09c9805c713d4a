// epilogue.hpp -- from the packed half-length spectrum to the output layouts.
//
// A real frame x[0..N) is transformed as one complex sequence of M = N/2
// points, z[n] = x[2n] + i x[2n+1].  With Z = DFT_M(z):
//     E[k] = (Z[k] + conj Z[M-k]) / 2          = DFT_M(x[0::2])[k]
//     O[k] = (Z[k] - conj Z[M-k]) / (2i)       = DFT_M(x[1::2])[k]
// The last radix-2 stage of the N-point transform is
//     X[k] = E[k] + W_N^k O[k],   X[k+M] = E[k] - W_N^k O[k],
// and the buffer one stage earlier -- what the reference returns for odd
// window exponents >= 13 -- is simply [E, O].  Either way bin k of the packed
// spectrum yields the outputs at positions k and M+k of the frame.
#pragma once

#include "engine.hpp"
#include "fft_device.hpp"

namespace ostft {

// Twice the outputs at positions k and M + k: the halvings of E and O are
// left to the output conversion (one exact scaling by a power of two there,
// folded into a constant for the real layouts), which saves vector ALU work.
struct BinPair {
    float2 lo;  // 2 X[k]
    float2 hi;  // 2 X[M + k]
};

// COMBINE: final radix-2 stage with w = W_N^k; otherwise [E, O]
template <bool COMBINE>
__device__ __forceinline__ BinPair finish_pair(float2 zk, float2 zm, float2 w)
{
    const float2 E = make_float2(zk.x + zm.x, zk.y - zm.y);  // 2 E
    const float2 O = make_float2(zk.y + zm.y, zm.x - zk.x);  // 2 O
    BinPair r;
    if constexpr (COMBINE) {
        const float2 t = cmul(w, O);
        r.lo = cadd(E, t);
        r.hi = csub(E, t);
    } else {
        r.lo = E;
        r.hi = O;
    }
    return r;
}

// the output conversions of a doubled value x2 = 2 X:
// sqrt(Re^2 + Re^2) of the Serial runner's ToPower, as sqrt(2)|Re|
__device__ __forceinline__ float compat_power(float2 x2)
{
    constexpr float HALF_SQRT2 = 1.41421356237309504880f * 0.5f;  // exactly half the float sqrt(2)
    return HALF_SQRT2 * fabsf(x2.x);
}
// |X| with the hardware square root (1 ulp)
// (fused multiply-adds written out, as in cmul)
__device__ __forceinline__ float magnitude(float2 x2)
{
    return 0.5f * __builtin_amdgcn_sqrtf(fmaf(x2.x, x2.x, x2.y * x2.y));
}
__device__ __forceinline__ float power_of(float2 x2) { return 0.25f * fmaf(x2.x, x2.x, x2.y * x2.y); }
__device__ __forceinline__ float2 value_of(float2 x2) { return make_float2(0.5f * x2.x, 0.5f * x2.y); }
__device__ __forceinline__ float2 conj_value_of(float2 x2) { return make_float2(0.5f * x2.x, -0.5f * x2.y); }

}  // namespace ostft
