// encode_field.hip -- the MATLAB toolbox's hologram encodings of a complex
// field on gfx950 (OpenHolo_Encoding/fn_encoding.m:1-98).
//
//   SSB         single sideband: centred spectrum, one half zeroed
//               (:29-47), inverse, real part scaled to [0, 1]
//   NI          numerical interference with a plane reference of amplitude
//               max|U| (:49-54), scaled by its maximum
//   P2A         angle(U) + pi/(2 pi) as the reference writes it (:56-58):
//               angle + 0.5
//   REAL        Re(U) (:20-21)
//   BURCKHARDT  three non-negative components per pixel (:60-83)
//   TWO_PHASE   two phases angle + pi +- acos(|U|/max|U|) per pixel (:85-98)
// The reference's quirks are kept: the sideband block starts at 1-based
// index floor(N/2) (so 'left' also drops the DC column and the one below
// it), P2A's operator precedence, and Burckhardt's second component of each
// branch without the amplitude factor.
//
// fftshift(fft2(ifftshift(.))) and its inverse on even sizes: the shifts
// are circular shifts by N/2, which the forward and inverse transforms
// undo between themselves, so SSB is IFFT(M FFT(U)) with the mask M in FFT
// order: 'left' zeroes frequencies -1 .. N/2-1 (FFT indices 0 .. N/2-1 and
// N-1), 'right' zeroes -N/2 .. -1 (indices N/2 .. N-1); 'top'/'bottom' the
// same on rows.
//
// The mask depends on one axis only, and the other axis's transform and its
// inverse cancel: 'left' and 'right' are a one-dimensional filter of every
// row, 'top' and 'bottom' of every column, one pass over the field (forward
// transform, mask and inverse transform of a line without leaving the
// workgroup) instead of four transforms and the masking.
//
// Reductions (max |U|^2, min/max of a float array) are exact in any order: a
// pass that needs one leaves a (min, max) pair per workgroup and the next pass
// starts by combining them, so every pass is one HBM sweep and one launch.
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <type_traits>

#include "fft_engine.h"
#include "fft_kernels.h"
#include "oph_internal.h"

namespace {

constexpr int RT = 256;      // threads per workgroup
constexpr int RB = 1024;     // workgroups of a reducing pass (and partial pairs), at most
constexpr int MB = 16384;    // workgroups of the other passes, at most

// (min, max) over the workgroup of each thread's (mn, mx); every thread of
// the workgroup calls it and gets the result.  NT threads, a multiple of 64
// or a power of two below it: there only the lanes that exist are exchanged
// (a shuffle reads 0 from one that does not).
template <int NT>
__device__ __forceinline__ float2 block_minmax(float mn, float mx) {
    static_assert(NT % 64 == 0 || (NT < 64 && (NT & (NT - 1)) == 0), "whole waves, or a power of two of lanes");
    __shared__ float2 w[(NT + 63) / 64];
#pragma unroll
    for (int o = (NT < 64 ? NT : 64) / 2; o > 0; o >>= 1) {
        mn = fminf(mn, __shfl_xor(mn, o, 64));
        mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    }
    __syncthreads();
    if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = make_float2(mn, mx);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < (NT + 63) / 64; ++k) {
        mn = fminf(mn, w[k].x);
        mx = fmaxf(mx, w[k].y);
    }
    return make_float2(mn, mx);
}

// (min, max) of the nb pairs an earlier pass left (RT threads)
__device__ __forceinline__ float2 combine(const float2* __restrict__ part, int nb) {
    float mn = FLT_MAX, mx = -FLT_MAX;
    for (int i = threadIdx.x; i < nb; i += RT) {
        const float2 p = part[i];
        mn = fminf(mn, p.x);
        mx = fmaxf(mx, p.y);
    }
    return block_minmax<RT>(mn, mx);
}

__global__ __launch_bounds__(RT) void abs2_minmax_partial(const float2* __restrict__ u, int64_t n, float2* part) {
    float mn = FLT_MAX, mx = -FLT_MAX;
    for (int64_t i = (int64_t)blockIdx.x * RT + threadIdx.x; i < n; i += (int64_t)gridDim.x * RT) {
        const float2 v = u[i];
        const float a = fmaf(v.x, v.x, v.y * v.y);
        mn = fminf(mn, a);
        mx = fmaxf(mx, a);
    }
    const float2 m = block_minmax<RT>(mn, mx);
    if (threadIdx.x == 0) part[blockIdx.x] = m;
}

// One-dimensional single-sideband filter of the lines of a field: columns
// (COLS; B neighbouring ones per workgroup, thread T of line T % B) or rows
// (B per workgroup, threads of a line side by side); the real part and each
// workgroup's (min, max).  A line that is not finite spoils the whole field,
// as it does in a two-dimensional transform: its (NaN, NaN) partial, which
// ssb_scale looks for, carries that over.
// Bound by HBM (8 bytes in, 4 out per pixel) and the transforms' LDS passes:
// 2048^2 rows 19 us; with ssb_scale 28 us a call, where four transforms, two
// copies, the masking, two reductions and the scaling took 115.
template <int L>
constexpr int ssb_lines(bool cols) { return cols ? fftk::col_lines(L) : fftk::row_lines(L); }

template <int L, bool COLS>
__global__ __launch_bounds__(ssb_lines<L>(COLS) * (L / 16)) void ssb_filter(const float2* __restrict__ u,
                                                                           float* __restrict__ out, int lines,
                                                                           int upper, float scale,
                                                                           const float2* __restrict__ tw,
                                                                           float2* part) {
    constexpr int TPL = L / 16, B = ssb_lines<L>(COLS), NT = B * TPL;
    constexpr int PL = COLS ? fft::skewed_len(L, B) : fft::padded_len(L);
    extern __shared__ float2 ssb_lds[];
    const int b = COLS ? threadIdx.x % B : threadIdx.x / TPL;
    const int t = COLS ? threadIdx.x / B : threadIdx.x % TPL;
    float2* buf = ssb_lds + b * PL;
    // (rows keep the twiddles in registers; a column workgroup is up to 1024
    // threads of 128 registers and reads them from the table at each stage)
    fft::Twiddles<COLS ? 16 : L> T;
    if constexpr (!COLS) T.load(tw, t);
    // element i of line l at l ls + i es
    const size_t ls = COLS ? 1 : L, es = COLS ? (size_t)lines : 1;
    float mn = FLT_MAX, mx = -FLT_MAX;
    bool nan = false;
    const int groups = (lines + B - 1) / B;
    for (int g0 = blockIdx.x; g0 < groups; g0 += gridDim.x) {
        const int l = (COLS ? xcd_remap(g0, groups) : g0) * B + b;
        const bool ok = l < lines;
        const size_t at = (size_t)(ok ? l : 0) * ls;
        float2 v[16];
#pragma unroll
        for (int m = 0; m < 16; ++m) v[m] = u[at + (size_t)(t + m * TPL) * es];
        // (a zero the compiler cannot see through: it would hoist the table
        // reads out of the loop into registers)
        int tz = t;
        if constexpr (COLS) asm volatile("" : "+v"(tz));
        auto line = [&](auto sign) {
            if constexpr (COLS) fft::line_regs_tw<L, sign>(v, buf, tw, tz);
            else fft::line_regs<L, sign>(v, buf, T, t);
        };
        __syncthreads();   // the previous line's last-stage reads are done
        line(std::integral_constant<int, -1>{});
#pragma unroll
        for (int m = 0; m < 16; ++m) {
            const int k = t + m * TPL;
            const bool stop = upper ? k >= L / 2 : k < L / 2 || k == L - 1;
            if (stop) v[m] = make_float2(0.f, 0.f);
        }
        __syncthreads();
        line(std::integral_constant<int, +1>{});
        if (!ok) continue;
#pragma unroll
        for (int m = 0; m < 16; ++m) {
            const float x = v[m].x * scale;
            out[at + (size_t)(t + m * TPL) * es] = x;
            mn = fminf(mn, x);
            mx = fmaxf(mx, x);
            nan |= !(fabsf(x) <= FLT_MAX);
        }
    }
    const float2 p = block_minmax<NT>(mn, mx);
    const bool bad = __syncthreads_or(nan);
    if (threadIdx.x == 0) part[blockIdx.x] = bad ? make_float2(NAN, NAN) : p;
}

// out = (v - min)/(max - min)  (SSB: realPositive / max(realPositive))
__global__ __launch_bounds__(RT) void ssb_scale(float* out, int64_t n, const float2* __restrict__ part, int nb) {
    bool nan = false;
    for (int i = threadIdx.x; i < nb; i += RT) nan |= part[i].x != part[i].x;
    const bool bad = __syncthreads_or(nan);
    const float2 m = combine(part, nb);
    for (int64_t i = (int64_t)blockIdx.x * RT + threadIdx.x; i < n; i += (int64_t)gridDim.x * RT)
        out[i] = bad ? NAN : (out[i] - m.x) / (m.y - m.x);
}

// NI first pass: |U + max|U||^2, and its (min, max) per workgroup
__global__ __launch_bounds__(RT) void ni_map(const float2* __restrict__ u, float* __restrict__ out, int64_t n,
                                             const float2* __restrict__ part2, int nb, float2* part) {
    const float ref = sqrtf(combine(part2, nb).y);
    float mn = FLT_MAX, mx = -FLT_MAX;
    for (int64_t i = (int64_t)blockIdx.x * RT + threadIdx.x; i < n; i += (int64_t)gridDim.x * RT) {
        const float2 v = u[i];
        const float re = v.x + ref;
        const float o = fmaf(re, re, v.y * v.y);
        out[i] = o;
        mn = fminf(mn, o);
        mx = fmaxf(mx, o);
    }
    const float2 m = block_minmax<RT>(mn, mx);
    if (threadIdx.x == 0) part[blockIdx.x] = m;
}

// out /= max(out)
__global__ __launch_bounds__(RT) void div_max(float* out, int64_t n, const float2* __restrict__ part, int nb) {
    const float mx = combine(part, nb).y;
    for (int64_t i = (int64_t)blockIdx.x * RT + threadIdx.x; i < n; i += (int64_t)gridDim.x * RT) out[i] = out[i] / mx;
}

__global__ void p2a_real_map(const float2* __restrict__ u, float* __restrict__ out, int64_t n, int p2a) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float2 v = u[i];
    out[i] = p2a ? atan2f(v.y, v.x) + 0.5f : v.x;
}

// Burckhardt (fn_encoding.m:60-83) and two-phase (:85-98), one pixel per
// thread and step (pixel i's components are out[3 i ..] and out[2 i ..]);
// the pairs hold max |U|^2.  angle(U/m) = angle(U) for m > 0.
__global__ __launch_bounds__(RT) void burckhardt_map(const float2* __restrict__ u, float* __restrict__ out, int64_t n,
                                                     const float2* __restrict__ part2, int nb) {
    const float m = sqrtf(combine(part2, nb).y);
    for (int64_t i = (int64_t)blockIdx.x * RT + threadIdx.x; i < n; i += (int64_t)gridDim.x * RT) {
        const float2 v = u[i];
        const float re = v.x / m, im = v.y / m;
        const float am = sqrtf(fmaf(re, re, im * im));
        const float ph = atan2f(im, re) + 3.14159265358979323846f;
        constexpr float third = 2.09439510239319549f, two_third = 4.18879020478639098f, two_pi = 6.28318530717958648f;
        constexpr float inv_s3 = 0.57735026918962576f;
        float a1 = 0.f, a2 = 0.f, a3 = 0.f;
        if (ph >= 0.f && ph < third) {
            a1 = am * (cosf(ph) + sinf(ph) * inv_s3);
            a2 = 2.f * sinf(ph) * inv_s3;
        } else if (ph >= third && ph < two_third) {
            const float q = ph - third;
            a2 = am * (cosf(q) + sinf(q) * inv_s3);
            a3 = 2.f * sinf(q) * inv_s3;
        } else if (ph >= two_third && ph < two_pi) {
            const float q = ph - two_third;
            a3 = am * (cosf(q) + sinf(q) * inv_s3);
            a1 = 2.f * sinf(q) * inv_s3;
        }
        out[3 * i] = a1;
        out[3 * i + 1] = a2;
        out[3 * i + 2] = a3;
    }
}

__global__ __launch_bounds__(RT) void two_phase_map(const float2* __restrict__ u, float* __restrict__ out, int64_t n,
                                                    const float2* __restrict__ part2, int nb) {
    const float m = sqrtf(combine(part2, nb).y);
    for (int64_t i = (int64_t)blockIdx.x * RT + threadIdx.x; i < n; i += (int64_t)gridDim.x * RT) {
        const float2 v = u[i];
        const float re = v.x / m, im = v.y / m;
        const float am = fminf(sqrtf(fmaf(re, re, im * im)), 1.f);
        const float ph = atan2f(im, re) + 3.14159265358979323846f;
        const float d = acosf(am);
        out[2 * i] = ph + d;
        out[2 * i + 1] = ph - d;
    }
}

template <int L, bool COLS>
int launch_ssb(oph_ctx* ctx, const float2* u, float* out, int lines, int upper, float2* part, int* nb) {
    const float2* tw = oph_twiddles(ctx, L);
    if (!tw) return OPH_ENOMEM;
    constexpr int B = ssb_lines<L>(COLS), NT = B * (L / 16);
    constexpr size_t shm = (size_t)B * (COLS ? fft::skewed_len(L, B) : fft::padded_len(L)) * sizeof(float2);
    static bool attr = false;
    if (!attr) {
        hipFuncSetAttribute(reinterpret_cast<const void*>(&ssb_filter<L, COLS>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
        hipGetLastError();
        attr = true;
    }
    *nb = std::min(RB, (lines + B - 1) / B);
    OPH_LAUNCH(ctx, "ssb_filter", (ssb_filter<L, COLS>), dim3(*nb), dim3(NT), shm, u, out, lines, upper,
               (float)(1.0 / (double)L), tw, part);
    return OPH_OK;
}

template <bool COLS>
int ssb_dispatch(oph_ctx* ctx, int L, const float2* u, float* out, int lines, int upper, float2* part, int* nb) {
    switch (L) {
#define OPH_SSB_CASE(n) \
    case n: return launch_ssb<n, COLS>(ctx, u, out, lines, upper, part, nb);
        OPH_FFT_LENGTHS(OPH_SSB_CASE)
#undef OPH_SSB_CASE
    }
    return oph_fail(ctx, OPH_ENOTSUP, "FFT length %d not supported (16..8192)", L);
}

}  // namespace

extern "C" int oph_encode_field(oph_ctx* ctx, const oph_c64* field, int nx, int ny, int method, int passband,
                                float* out, int flags) {
    int rc = oph_enter(ctx);
    if (rc) return rc;
    if (!field || !out || nx <= 0 || ny <= 0) return oph_fail(ctx, OPH_EINVAL, "bad encode arguments");
    if (method < OPH_ENC_SSB || method > OPH_ENC_TWO_PHASE) return oph_fail(ctx, OPH_EINVAL, "unknown method %d", method);
    if (method == OPH_ENC_SSB) {
        if (passband < OPH_PASS_LEFT || passband > OPH_PASS_BOTTOM)
            return oph_fail(ctx, OPH_EINVAL, "unknown passband %d", passband);
        if (!fftk::supported(nx) || !fftk::supported(ny))
            return oph_fail(ctx, OPH_ENOTSUP, "SSB size %dx%d: each side must be a power of two in 16..8192", nx, ny);
    }
    if ((flags & OPH_ASYNC) && !(flags & OPH_DEVICE_PTR))
        return oph_fail(ctx, OPH_EINVAL, "OPH_ASYNC needs device pointers");
    const int64_t n = (int64_t)nx * ny;
    const int64_t nout = n * (method == OPH_ENC_BURCKHARDT ? 3 : method == OPH_ENC_TWO_PHASE ? 2 : 1);
    const float2* u = reinterpret_cast<const float2*>(field);
    float* o = out;
    if (!(flags & OPH_DEVICE_PTR)) {
        float2* du = static_cast<float2*>(oph_scratch(ctx, SLOT_IN, n * sizeof(float2)));
        o = static_cast<float*>(oph_scratch(ctx, SLOT_OUT, nout * sizeof(float)));
        if (!du || !o) return OPH_ENOMEM;
        OPH_HIP_CHECK(ctx, hipMemcpyAsync(du, field, n * sizeof(float2), hipMemcpyHostToDevice, ctx->stream));
        u = du;
    }
    // two reductions' pairs (NI reads the first's during the second)
    float2* part = static_cast<float2*>(oph_scratch(ctx, SLOT_AUX1, sizeof(float2) * 2 * RB));
    if (!part) return OPH_ENOMEM;
    float2* part2 = part + RB;
    int nb = (int)std::min<int64_t>(RB, (n + RT - 1) / RT);
    const dim3 grid(nb), blk(RT);
    // passes without a reduction of their own (each workgroup first combines
    // the pairs): eight pixels a thread, fewer while that leaves the chip idle
    // (Burckhardt: 1024 x 512 11.6 us at two, 15.2 at eight; 4096^2 120 us at
    // eight, 137 in 1,024 workgroups of 64)
    const dim3 mgrid((unsigned)std::min<int64_t>(MB, std::max<int64_t>(nb, (n + 8 * RT - 1) / (8 * RT))));
    if (method != OPH_ENC_SSB && method != OPH_ENC_P2A && method != OPH_ENC_REAL)
        OPH_LAUNCH(ctx, "abs2_minmax_partial", abs2_minmax_partial, grid, blk, 0, u, n, part);
    switch (method) {
        case OPH_ENC_SSB: {
            const int upper = passband == OPH_PASS_RIGHT || passband == OPH_PASS_BOTTOM;
            int np = 0;
            if (reinterpret_cast<const char*>(u) < reinterpret_cast<const char*>(o + n) &&
                reinterpret_cast<const char*>(o) < reinterpret_cast<const char*>(u + n)) {
                // out overlaps the field, which the filter still reads while it writes
                float2* w = static_cast<float2*>(oph_scratch(ctx, SLOT_WORK0, n * sizeof(float2)));
                if (!w) return OPH_ENOMEM;
                OPH_HIP_CHECK(ctx, hipMemcpyAsync(w, u, n * sizeof(float2), hipMemcpyDeviceToDevice, ctx->stream));
                u = w;
            }
            rc = passband == OPH_PASS_LEFT || passband == OPH_PASS_RIGHT
                     ? ssb_dispatch<false>(ctx, nx, u, o, ny, upper, part, &np)
                     : ssb_dispatch<true>(ctx, ny, u, o, nx, upper, part, &np);
            if (rc) return rc;
            OPH_LAUNCH(ctx, "ssb_scale", ssb_scale, mgrid, blk, 0, o, n, part, np);
            break;
        }
        case OPH_ENC_NI:
            OPH_LAUNCH(ctx, "ni_map", ni_map, grid, blk, 0, u, o, n, part, nb, part2);
            OPH_LAUNCH(ctx, "div_max", div_max, mgrid, blk, 0, o, n, part2, nb);
            break;
        case OPH_ENC_P2A:
        case OPH_ENC_REAL:
            OPH_LAUNCH(ctx, "p2a_real_map", p2a_real_map, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, u, o, n,
                       method == OPH_ENC_P2A ? 1 : 0);
            break;
        case OPH_ENC_BURCKHARDT:
            OPH_LAUNCH(ctx, "burckhardt_map", burckhardt_map, mgrid, blk, 0, u, o, n, part, nb);
            break;
        default:
            OPH_LAUNCH(ctx, "two_phase_map", two_phase_map, mgrid, blk, 0, u, o, n, part, nb);
            break;
    }
    if (!(flags & OPH_DEVICE_PTR))
        OPH_HIP_CHECK(ctx, hipMemcpyAsync(out, o, nout * sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
    return oph_finish(ctx, flags);
}
