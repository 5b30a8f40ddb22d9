// pa_selftest.hip -- device halves of the engine's self-tests (pa_selftest): small kernels that run
// the production device functions (pa_device.hpp) on the closed-form inputs of the reference's
// unit tests (PrivacyAmplification.cu:299-737).  The rest of each test drives the production
// kernels themselves through their launchers (pa_engine.cpp).
#include <hip/hip_runtime.h>

#include "pa_device.hpp"
#include "pa_geom.hpp"
#include "pa_kernels.hpp"

namespace pa {

// out[i] = correction(wk[i], ws[i], L): the correction term exactly as k_small computes it
// (unitTestCalculateCorrectionFloat's inputs, PrivacyAmplification.cu:299-361).
__global__ __launch_bounds__(256) void k_st_correction(const uint32_t* __restrict__ wk, const uint32_t* __restrict__ ws,
                                                       uint32_t L, float* __restrict__ out, uint32_t count) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i < count) out[i] = correction(wk[i], ws[i], L);
}

// The spectral product as the row pass forms it: the complex product of the key's and the seed's
// values (ElementWiseProduct, PrivacyAmplification.cu:465-481, with its 1/r pre-scaling applied to
// both operands as the reference does), and the round trip of the real-FFT splits that surround it
// in k_small: c2r_split(r2c_split(z)) = 4 z for every partner pair (k, N-k).
__global__ __launch_bounds__(256) void k_st_product(const float2* __restrict__ a, const float2* __restrict__ b,
                                                    float r, float2* __restrict__ prod, const float2* __restrict__ z,
                                                    float2* __restrict__ zz, uint32_t N) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i < N) {
        const float inv = 1.0f / r;
        prod[i] = cmul(cscale(a[i], inv), cscale(b[i], inv));
    }
    if (i >= 1 && i < N / 2) {  // pair (i, N - i), split twiddle w = exp(-2 pi i i / (2N))
        const double ang = -3.14159265358979323846 * (double)i / (double)N;
        const float2 w = make_float2((float)cos(ang), (float)sin(ang));
        const float2 wp = make_float2(-w.x, w.y);  // the partner's: -conj(w)
        const float2 xk = r2c_split(z[i], z[N - i], w), xp = r2c_split(z[N - i], z[i], wp);
        zz[i] = c2r_split(xk, xp, w);
        zz[N - i] = c2r_split(xp, xk, wp);
    }
}

// Pass A' output for the ToBinaryArray closed form (PrivacyAmplification.cu:669-737): the
// pre-rounding value of conv index p is v[p] = bit 31 - (p mod 32) of the integer p / 32 (0 or 1);
// the pieces hold round_bit(v * invN + corr) of their positions, in pass A''s layout: bit e of
// piece[(half N2 + t2) N1/16 + j] is position half N + t2 + N2 (j + (N1/16) e).
__device__ __forceinline__ float st_pattern(uint32_t p) { return (float)(((p >> 5) >> (31u - (p & 31u))) & 1u); }
__global__ __launch_bounds__(256) void k_st_pieces(uint16_t* __restrict__ piece, Geom g, float corr, float invN) {
    const uint64_t e = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    if (e >= (uint64_t)g.L / 16) return;
    const uint32_t S = g.N1 / 16u, j = (uint32_t)(e % S), ht = (uint32_t)(e / S);  // ht = half N2 + t2
    const uint32_t p0 = (ht / g.N2) * g.N + ht % g.N2 + g.N2 * j;
    float dist = 0.f;
    uint32_t bits = 0;
    for (uint32_t k = 0; k < 16; ++k) bits |= round_bit(st_pattern(p0 + g.N2 * S * k) * invN + corr, dist) << k;
    piece[e] = (uint16_t)bits;
}

hipError_t launch_st_correction(const uint32_t* wk, const uint32_t* ws, uint32_t L, float* out, uint32_t count,
                                hipStream_t s) {
    k_st_correction<<<(count + 255u) / 256u, 256, 0, s>>>(wk, ws, L, out, count);
    return hipGetLastError();
}
hipError_t launch_st_product(const float2* a, const float2* b, float r, float2* prod, const float2* z, float2* zz,
                             uint32_t N, hipStream_t s) {
    k_st_product<<<(N + 255u) / 256u, 256, 0, s>>>(a, b, r, prod, z, zz, N);
    return hipGetLastError();
}
hipError_t launch_st_pieces(uint8_t* nib, const Geom& g, float corr, float invN, hipStream_t s) {
    k_st_pieces<<<g.L / 16u / 256u, 256, 0, s>>>(reinterpret_cast<uint16_t*>(nib), g, corr, invN);
    return hipGetLastError();
}

}  // namespace pa
