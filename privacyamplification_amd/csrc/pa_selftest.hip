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

// Pass B's output R' for the ToBinaryArray closed form (PrivacyAmplification.cu:669-737): column t2 is
// cols[(t2 - c0) N1 + k1] for c0 <= t2 < c0 + nc, else base[k1] times c's component t2 mod 4; in pass A''s
// tiles where they are used.
__global__ __launch_bounds__(256) void k_st_rows(float2* __restrict__ R, Geom g, const float2* __restrict__ base, float4 c,
                                                 const float2* __restrict__ cols, uint32_t c0, uint32_t nc) {
    const uint32_t e = blockIdx.x * 256u + threadIdx.x;
    if (e >= g.N) return;
    const uint32_t k1 = e / g.N2, t2 = e % g.N2, r = t2 & 3u;
    const float2 v = t2 >= c0 && t2 - c0 < nc ? cols[(size_t)(t2 - c0) * g.N1 + k1]
                                              : cscale(base[k1], r == 0u ? c.x : r == 1u ? c.y : r == 2u ? c.z : c.w);
    R[rt_tiled(g.lg1) ? ((size_t)(t2 / RT_COLS) * g.N1 + k1) * RT_COLS + t2 % RT_COLS : (size_t)e] = v;
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
hipError_t launch_st_rows(float2* R, const Geom& g, const float2* base, float4 c, const float2* cols, uint32_t c0,
                          uint32_t nc, hipStream_t s) {
    k_st_rows<<<(g.N + 255u) / 256u, 256, 0, s>>>(R, g, base, c, cols, c0, nc);
    return hipGetLastError();
}

}  // namespace pa
