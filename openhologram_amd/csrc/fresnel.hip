// fresnel.hip -- Fresnel point-cloud hologram on gfx950: the separable form of
// the sum as an MFMA complex contraction in FP32, FP16 or BF16.
//
// Field (the direct Fresnel sum of CWO/cwoPLS.cpp:370-422, with the point
// amplitude, its initial phase and the plane carrier exp(i k z_n)):
//   U[i][j] = sum_n a_n exp(i (k z_n + phi_n)) exp(i k ((X_j - x_n)^2 + (Y_i - y_n)^2) / (2 z_n))
//   X_j = (j - nx/2) p,  Y_i = (i - ny/2) p                 (cwoPLS.cpp:400-401)
// The quadratic phase separates, exp(i k (dx^2 + dy^2)/(2z)) =
// exp(i k dx^2/(2z)) exp(i k dy^2/(2z)), so U = A B^T with
//   A[i][n] = w_n exp(i pi (Y_i - y_n)^2/(lambda z_n)),  B[j][n] = exp(i pi (X_j - x_n)^2/(lambda z_n)),
//   w_n = a_n exp(i (k z_n + phi_n)):
// a complex (pixels x points)(points x pixels) contraction.  The chirp phases
// reach ~1e4 turns and are reduced in FP64 before the FP32 sin/cos; the
// factors are rounded to BF16 or FP16, optionally split as hi + lo (the lo
// part carries the rounding error of hi), and contracted on MFMA with FP32
// accumulation (A B = Ah Bh + Ah Bl + Al Bh).
#include <algorithm>
#include <cmath>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include "oph_internal.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

namespace {

struct FrPoint {
    double x, y, c;   // position, c = 1/(2 lambda z) (turns per m^2)
    float wre, wim;   // a exp(i 2 pi frac(z/lambda + phi/2pi))
    float f0, a;      // frac(z/lambda + phi/2pi), amplitude
};

__device__ FrPoint make_frpoint(const double* x, const double* y, const double* z, const double* amp,
                                const double* phase, int64_t i, double lambda) {
    FrPoint q;
    q.x = x[i];
    q.y = y[i];
    q.c = 1.0 / (2.0 * lambda * z[i]);
    double t = z[i] / lambda + (phase ? phase[i] * 0.15915494309189535 : 0.0);
    t -= rint(t);
    const float a = amp ? (float)amp[i] : 1.f;
    q.f0 = (float)t;
    q.a = a;
    q.wre = a * cos_turns((float)t);
    q.wim = a * sin_turns((float)t);
    return q;
}

// a zero-weight point (padding up to whole contraction chunks) on plane c
__device__ FrPoint zero_frpoint(double c) {
    FrPoint q;
    q.x = q.y = 0.0;
    q.c = c;
    q.f0 = 0.f;
    q.a = 0.f;
    q.wre = q.wim = 0.f;
    return q;
}

// skip: when set and *skip != 0 the plane-factored form computes the field
// and this general preparation (and contraction) does nothing
__global__ void fresnel_prep(const double* x, const double* y, const double* z, const double* amp,
                             const double* phase, int64_t n, int64_t npad, double lambda, FrPoint* out,
                             const int* skip) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= npad || (skip && *skip)) return;
    out[i] = i < n ? make_frpoint(x, y, z, amp, phase, i, lambda) : zero_frpoint(0.0);
}

// ---------------------------------------------------------------------------
// FP32 contraction (OPH_FRESNEL_VALU): the separable form U = A B^T with the
// chirp factors in FP32 (phases reduced in FP64) on v_mfma_f32_32x32x2_f32.
// A workgroup of 4 waves owns a 64 x 128 pixel tile; each wave contracts 32
// rows x 64 columns.  The points come in chunks of F32_PTS: while a chunk is
// contracted from one LDS buffer the next one's factors are generated into
// the other (a lane owns one row or column, each wave a quarter of the
// points, whose records are wave-uniform), one barrier per chunk.  A factor
// costs one FP64 phase and one sin/cos for every row and column of the tile
// instead of one per pixel: 192 per point and 8,192 pixels.  Sums run in FP32
// over F32_BATCH points and in FP64 across batches, so a pixel's rounding
// error does not grow with the point count.
//
// The complex product takes three real ones (sums of A.x B.x, A.y B.y and
// (A.x + A.y)(B.x + B.y)): a quarter fewer matrix instructions; the sums'
// rounding grows by 1.4, which the short batches make up for.
//
// Error against FP64 in the 2-norm: 2.4e-7 from some 300 points on, at any
// distance from 20 mm to 2 m (batches of 128: 3.1e-7, of 256: 4.2e-7, of 32:
// 1.9e-7); 2.2e-7 at 100 points, 1.3e-7 to 1.5e-7 at one, the rounding of two
// factors of a phase, a sin and a cos each.  A sum per pixel on the vector
// unit had 4.3e-7 at 0.1 m, 1.5e-6 at 20 mm and 3.0e-7 to 3.2e-7 beyond 0.3 m
// (there 2.0e-7 at 100 points, 1.0e-7 at one, which two factors cannot reach).
//
// Bound by the matrix cores (96 cycles per point and 32 x 32 pixels) and, as
// vector and matrix instructions do not overlap on a SIMD here, by the
// generation in turn with them: 1280 x 720 with 20,000 points 1.16 ms (before
// the test for huge amplitudes 1.14, with batches of 256 1.08, of 128 1.10, of
// 32 1.20; 1.30 with four products and
// batches of 256, of which the generation is 0.16; interleaving the two
// instruction by instruction changed nothing).  A sum per pixel took 4.95 ms.

constexpr int F32_PTS = 16, F32_BATCH = 64;
constexpr int F32_R = 64, F32_C = 128;

// An amplitude so large that products of its factors may overflow where the
// point's own value does not (or infinite, or NaN: inf - inf in the three sums
// would be NaN where the point adds +-inf).  Such points are left out of the
// contraction and added per pixel.
__device__ __forceinline__ bool f32_huge(float a) {
    return (__builtin_bit_cast(unsigned, a) & 0x7FFFFFFFu) > 0x7149F2CAu;   // 1e30
}

struct F32Args {
    const FrPoint* pts;
    int64_t npad, chunk;   // multiples of KC
    int nx, ny;
    double p;
    float2* out;           // [chunks][ny][nx]
};

struct F32Lds {
    float2 A[F32_PTS][F32_R];
    float2 B[F32_PTS][F32_C];
};

__global__ __launch_bounds__(256, 2) void fresnel_f32(F32Args a) {
    __shared__ F32Lds lds[2];
    __shared__ int any_huge;
    const int lane = threadIdx.x & 63;
    if (threadIdx.x == 0) any_huge = 0;
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row0 = blockIdx.y * F32_R, col0 = blockIdx.x * F32_C;
    const double Y = (row0 + lane - a.ny / 2) * a.p;
    const double X0 = (col0 + lane - a.nx / 2) * a.p, X1 = (col0 + 64 + lane - a.nx / 2) * a.p;
    const int64_t pb = (int64_t)blockIdx.z * a.chunk;
    const int nch = (int)((min(a.npad, pb + a.chunk) - pb) / F32_PTS);

    // this wave's quarter of chunk c: the records (wave-uniform, by scalar
    // loads), then one point's factors (k) into L
    constexpr int PW = F32_PTS / 4;
    typedef const __attribute__((address_space(4))) FrPoint* PtsPtr;
    struct { double x, y, c; float f0, a; } q[PW];
    auto records = [&](int c) {
        PtsPtr p = (PtsPtr)(uintptr_t)(a.pts + pb + (int64_t)c * F32_PTS + wave * PW);
#pragma unroll
        for (int k = 0; k < PW; ++k) {
            q[k].x = p[k].x;
            q[k].y = p[k].y;
            q[k].c = p[k].c;
            q[k].f0 = p[k].f0;
            q[k].a = p[k].a;
        }
    };
    auto generate = [&](F32Lds& L) {
#pragma unroll
        for (int k = 0; k < PW; ++k) {
            const int pt = wave * PW + k;
            if (f32_huge(q[k].a)) {   // (the same for the whole wave)
                any_huge = 1;
                q[k].a = 0.f;
            }
            const double dy = Y - q[k].y, d0 = X0 - q[k].x, d1 = X1 - q[k].x;
            const float ty = (float)frac_turns(fma(q[k].c, dy * dy, (double)q[k].f0));
            const float t0 = (float)frac_turns(q[k].c * (d0 * d0)), t1 = (float)frac_turns(q[k].c * (d1 * d1));
            L.A[pt][lane] = make_float2(q[k].a * cos_turns(ty), q[k].a * sin_turns(ty));
            L.B[pt][lane] = make_float2(cos_turns(t0), sin_turns(t0));
            L.B[pt][64 + lane] = make_float2(cos_turns(t1), sin_turns(t1));
        }
    };

    f32x16 s1[2], s2[2], s3[2];   // sums of A.x B.x, A.y B.y, (A.x + A.y)(B.x + B.y)
    double sre[2][16], sim[2][16];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        s1[b] = s2[b] = s3[b] = (f32x16)0.f;
#pragma unroll
        for (int v = 0; v < 16; ++v) sre[b][v] = sim[b][v] = 0.0;
    }
    const int wr = 32 * (wave & 1), wc = 64 * (wave >> 1);
    if (nch > 0) {
        records(0);
        generate(lds[0]);
    }
    for (int c = 0; c < nch; ++c) {
        // (the last chunk generates itself once more, into the idle buffer)
        records(min(c + 1, nch - 1));
        __syncthreads();   // chunk c is complete; the other buffer's readers are done
        const F32Lds& L = lds[c & 1];
        F32Lds& N = lds[(c + 1) & 1];
        generate(N);
#pragma unroll
        for (int k = 0; k < F32_PTS; k += 2) {
            const int pt = k + (lane >> 5);
            const float2 A = L.A[pt][wr + (lane & 31)];
            float2 B[2];
#pragma unroll
            for (int b = 0; b < 2; ++b) B[b] = L.B[pt][wc + 32 * b + (lane & 31)];
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                s1[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(A.x, B[b].x, s1[b], 0, 0, 0);
                s2[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(A.y, B[b].y, s2[b], 0, 0, 0);
                s3[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(A.x + A.y, B[b].x + B[b].y, s3[b], 0, 0, 0);
            }
        }
        if ((c + 1) % (F32_BATCH / F32_PTS) == 0 || c + 1 == nch) {
#pragma unroll
            for (int b = 0; b < 2; ++b) {
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    sre[b][v] += (double)(s1[b][v] - s2[b][v]);
                    sim[b][v] += (double)(s3[b][v] - (s1[b][v] + s2[b][v]));
                }
                s1[b] = s2[b] = s3[b] = (f32x16)0.f;
            }
        }
    }
    __syncthreads();
    if (any_huge)
        for (int i = 0; i < nch * F32_PTS; ++i) {
            const FrPoint h = a.pts[pb + i];
            if (!f32_huge(h.a)) continue;
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const double dx = (col0 + wc + 32 * b + (lane & 31) - a.nx / 2) * a.p - h.x;
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const double dy = (row0 + wr + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3) - a.ny / 2) * a.p - h.y;
                    const float t = (float)frac_turns(fma(h.c, fma(dx, dx, dy * dy), (double)h.f0));
                    sre[b][v] += (double)(h.a * cos_turns(t));
                    sim[b][v] += (double)(h.a * sin_turns(t));
                }
            }
        }
    // register v of a lane: row 8 (v/4) + 4 (lane/32) + v%4, column lane%32
    float2* dst = a.out + (size_t)blockIdx.z * a.nx * a.ny;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const int col = col0 + wc + 32 * b + (lane & 31);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int row = row0 + wr + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
            if (row < a.ny && col < a.nx)
                dst[(size_t)row * a.nx + col] = make_float2((float)sre[b][v], (float)sim[b][v]);
        }
    }
}

__global__ void fresnel_sum_chunks(const float2* partial, int chunks, int64_t npix, float2* out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= npix) return;
    double re = 0.0, im = 0.0;
    for (int c = 0; c < chunks; ++c) {
        const float2 v = partial[(size_t)c * npix + i];
        re += v.x;
        im += v.y;
    }
    out[i] = make_float2((float)re, (float)im);
}

// ---------------------------------------------------------------------------
// MFMA contraction.  A workgroup of 8 waves owns a 256 x 128 output tile
// (256 rows of y, 128 columns of x); for each chunk of 32 points it writes
// the chirp factors A (256 rows) and B (128 columns) to LDS as 16-bit planes
// [re_hi, im_hi, re_lo, im_lo] laid out [row][point] (generated by a phase
// recurrence, below), then each wave contracts a 64 x 64 sub-tile with
// v_mfma_f32_32x32x16 (lane l supplies row l%32, points 8(l/32)..+7 of A and
// column l%32, the same points of B; accumulator register v of lane l is
// output row 8(v/4) + 4(l/32) + v%4, column l%32).  A chirp entry is
// generated once per tile and used by every output of its row or column, so
// the taller tile spends 3/4 of the generation per output of a square
// 128 x 128 one; the workgroup takes the whole CU (two waves per SIMD).

constexpr int MR = 256;         // output tile rows
constexpr int MC = 128;         // output tile columns
constexpr int KC = 32;          // padding granularity: the largest chunk
// points per chunk: 32 for the single-precision forms; 16 for the hi+lo
// forms, whose four operand planes in two buffers would not fit LDS at 32
template <bool SPLIT>
constexpr int KCH = SPLIT ? 16 : 32;
constexpr int MFMA_THREADS = 512;

template <typename T>
struct Mfma;

template <>
struct Mfma<__bf16> {
    typedef bf16x8 V;
    static __device__ __forceinline__ __bf16 cvt(float f) { return (__bf16)f; }
    // both parts in one packed conversion (round to nearest even)
    static __device__ __forceinline__ void cvt2(float re, float im, __bf16& rh, __bf16& ih) {
        const f32x2 v = {re, im};
        const bf16x2 h = __builtin_convertvector(v, bf16x2);
        rh = h.x;
        ih = h.y;
    }
    static __device__ __forceinline__ float back(__bf16 h) { return (float)h; }
    // the low parts (re - rh, im - ih, exact in FP32) in one packed conversion
    static __device__ __forceinline__ void lo2(float re, float im, __bf16 rh, __bf16 ih, float, __bf16& rl,
                                               __bf16& il) {
        cvt2(re - (float)rh, im - (float)ih, rl, il);
    }
    static __device__ __forceinline__ f32x16 mac(V a, V b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
};

template <>
struct Mfma<_Float16> {
    typedef f16x8 V;
    static __device__ __forceinline__ _Float16 cvt(float f) { return (_Float16)f; }
    static __device__ __forceinline__ void cvt2(float re, float im, _Float16& rh, _Float16& ih) {
        const f32x2 v = {re, im};
        const f16x2 h = __builtin_convertvector(v, f16x2);
        rh = h.x;
        ih = h.y;
    }
    static __device__ __forceinline__ float back(_Float16 h) { return (float)h; }
    // f - h rounded to FP16 (exact in FP32 before the rounding) as
    // f + h m1 with m1 = -1 from a register (a literal -1 would fold the FMA
    // into a subtraction): one mixed-precision FMA, FP16 operand widened
    static __device__ __forceinline__ _Float16 lo(float f, _Float16 h, float m1) {
        return (_Float16)fmaf((float)h, m1, f);
    }
    static __device__ __forceinline__ void lo2(float re, float im, _Float16 rh, _Float16 ih, float m1, _Float16& rl,
                                               _Float16& il) {
        rl = lo(re, rh, m1);
        il = lo(im, ih, m1);
    }
    static __device__ __forceinline__ f32x16 mac(V a, V b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
};

// two 16-bit values as one word, the first in the low half
template <typename T>
__device__ __forceinline__ unsigned pack2(T lo, T hi) {
    return (unsigned)__builtin_bit_cast(unsigned short, lo) | ((unsigned)__builtin_bit_cast(unsigned short, hi) << 16);
}

template <typename V>
__device__ __forceinline__ V negate(V v) {
    u32x4 u = __builtin_bit_cast(u32x4, v);
    u ^= 0x80008000u;
    return __builtin_bit_cast(V, u);
}

struct MfmaArgs {
    const FrPoint* pts;
    int64_t npad;     // multiple of KC
    int nx, ny;
    double p;
    float2* out;
    const int* skip;  // when set and nonzero, the plane-factored form has the field
};

template <typename T, bool SPLIT>
struct FrLds {
    static constexpr int NP = SPLIT ? 4 : 2;
    static constexpr int KS = KCH<SPLIT> + 8;   // row stride (elements): 16-byte aligned rows
    T A[NP][MR][KS];
    T B[NP][MC][KS];
};

// Chirp factors by a phase recurrence.  A run is one point's entries on
// rows (A, with the point weight) or columns (B) gph + G m, G = 32.  Along a
// run the phase c (Y - y)^2 has constant second difference
// delta = 2 c (G p)^2, so with R = exp(i 2 pi (phi_{m+1} - phi_m)),
// A_{m+1} = A_m R_m and R_{m+1} = R_m exp(i 2 pi delta): two complex
// multiplies per entry; the anchor phi_0, the first step and delta are
// reduced in FP64 once per run (phases of ~1e4 turns).  In the
// plane-factored form (below) the factor is geometric: one multiply.
// FULL: every row and column of the tile is inside the image (no per-entry
// bounds select).
//
// Two neighbouring points per thread: a thread runs points k and k + 1 over
// the same rows, so each operand plane takes one 32-bit LDS store per row
// (both points' 16-bit parts) instead of two 16-bit stores.  The generation
// is bound by the LDS store instructions, not by its arithmetic; the extra
// FP64 set-up of the second run is the cheaper side.
constexpr int GPH2 = 32;   // run stride with point pairs

template <typename T, bool SPLIT, bool FULL, int AB, bool PLANE, typename Args>
__device__ __forceinline__ void fr_run_pair(FrLds<T, SPLIT>& L, const double* p_x, const double* p_y,
                                            const double* p_c, const float* p_wr, const float* p_wi, int k, int gph,
                                            int i0, int j0, const Args& a) {
    constexpr int M = (AB == 0 ? MR : MC) / GPH2;
    constexpr int KS = FrLds<T, SPLIT>::KS;
    constexpr int PS = (AB == 0 ? MR : MC) * KS / 2;   // plane stride in 32-bit words
    const double sp = (double)GPH2 * a.p;
    const double P0 = AB == 0 ? (i0 + gph - a.ny / 2) * a.p : (j0 + gph - a.nx / 2) * a.p;
    float2 v[2], R[2], E[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const double c = p_c[k + h];
        const double u = AB == 0 ? p_y[k + h] : p_x[k + h];
        double t0, t1;
        if constexpr (PLANE) {
            // the plane's factor: phase c (u^2 - 2 P u), step -2 c u G p
            t0 = c * u * (u - 2.0 * P0);
            t1 = -2.0 * c * u * sp;
        } else {
            // the full chirp: phase c d^2, first step c (2 d G p + (G p)^2),
            // second difference 2 c (G p)^2
            const double d0 = P0 - u;
            t0 = c * d0 * d0;
            t1 = c * (2.0 * d0 * sp + sp * sp);
            double td = 2.0 * c * sp * sp;
            td -= rint(td);
            E[h] = make_float2(cos_turns((float)td), sin_turns((float)td));
        }
        t0 -= rint(t0);
        t1 -= rint(t1);
        v[h] = make_float2(cos_turns((float)t0), sin_turns((float)t0));
        if constexpr (AB == 0) {
            const float wr_ = p_wr[k + h], wi_ = p_wi[k + h];
            v[h] = make_float2(wr_ * v[h].x - wi_ * v[h].y, wr_ * v[h].y + wi_ * v[h].x);
        }
        R[h] = make_float2(cos_turns((float)t1), sin_turns((float)t1));
    }
    const int lim = AB == 0 ? a.ny - i0 : a.nx - j0;   // rows / columns inside the image
    unsigned* p0 = reinterpret_cast<unsigned*>(AB == 0 ? &L.A[0][gph][k] : &L.B[0][gph][k]);
    float m1 = -1.f;
    if constexpr (SPLIT) asm volatile("v_mov_b32 %0, -1.0" : "=v"(m1));
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const bool ok = FULL || gph + GPH2 * m < lim;
        float re[2], im[2];
        T rh[2], ih[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            re[h] = ok ? v[h].x : 0.f;
            im[h] = ok ? v[h].y : 0.f;
        }
        Mfma<T>::cvt2(re[0], re[1], rh[0], rh[1]);
        Mfma<T>::cvt2(im[0], im[1], ih[0], ih[1]);
        unsigned* q = p0 + m * GPH2 * KS / 2;
        q[0] = pack2(rh[0], rh[1]);
        q[PS] = pack2(ih[0], ih[1]);
        if constexpr (SPLIT) {
            T rl[2], il[2];
            Mfma<T>::lo2(re[0], re[1], rh[0], rh[1], m1, rl[0], rl[1]);
            Mfma<T>::lo2(im[0], im[1], ih[0], ih[1], m1, il[0], il[1]);
            q[2 * PS] = pack2(rl[0], rl[1]);
            q[3 * PS] = pack2(il[0], il[1]);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            v[h] = make_float2(fmaf(v[h].x, R[h].x, -v[h].y * R[h].y), fmaf(v[h].x, R[h].y, v[h].y * R[h].x));
            if constexpr (!PLANE)
                R[h] = make_float2(fmaf(R[h].x, E[h].x, -R[h].y * E[h].y), fmaf(R[h].x, E[h].y, R[h].y * E[h].x));
        }
    }
}

// One thread per (point pair, phase) -- or, with 16-point chunks, per
// (point pair, phase, factor): the first four waves take the A runs and the
// last four the B runs, one of each per SIMD.
template <typename T, bool SPLIT, bool FULL, bool PLANE, typename Args>
__device__ __forceinline__ void fr_generate_pairs(FrLds<T, SPLIT>& L, const double* p_x, const double* p_y,
                                                  const double* p_c, const float* p_wr, const float* p_wi, int tid,
                                                  int i0, int j0, const Args& a) {
    constexpr int NPAIR = KCH<SPLIT> / 2;
    if constexpr (!SPLIT) {
        static_assert(NPAIR * GPH2 == MFMA_THREADS, "one thread per (point pair, phase)");
        const int k = 2 * (tid % NPAIR), gph = tid / NPAIR;
        fr_run_pair<T, SPLIT, FULL, 0, PLANE>(L, p_x, p_y, p_c, p_wr, p_wi, k, gph, i0, j0, a);
        fr_run_pair<T, SPLIT, FULL, 1, PLANE>(L, p_x, p_y, p_c, p_wr, p_wi, k, gph, i0, j0, a);
    } else {
        static_assert(2 * NPAIR * GPH2 == MFMA_THREADS, "one thread per (point pair, phase, factor)");
        const int h = tid % (MFMA_THREADS / 2);
        const int k = 2 * (h % NPAIR), gph = h / NPAIR;
        if (tid < MFMA_THREADS / 2)
            fr_run_pair<T, SPLIT, FULL, 0, PLANE>(L, p_x, p_y, p_c, p_wr, p_wi, k, gph, i0, j0, a);
        else
            fr_run_pair<T, SPLIT, FULL, 1, PLANE>(L, p_x, p_y, p_c, p_wr, p_wi, k, gph, i0, j0, a);
    }
}

// Contraction of one chunk from L by wave (wr, wc): its 64 x 64 sub-tile.
template <typename T, bool SPLIT>
__device__ __forceinline__ void fr_contract(const FrLds<T, SPLIT>& L, int wr, int wc, int lane, f32x16 (&cr)[2][2],
                                            f32x16 (&ci)[2][2]) {
    typedef typename Mfma<T>::V V;
    constexpr int NP = FrLds<T, SPLIT>::NP;
#pragma unroll
    for (int s = 0; s < KCH<SPLIT> / 16; ++s) {
        const int kb = 16 * s + 8 * (lane >> 5);
        V A[2][NP], B[2][NP];
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            const int row = wr * 64 + 32 * x + (lane & 31);
            const int col = wc * 64 + 32 * x + (lane & 31);
#pragma unroll
            for (int q = 0; q < NP; ++q) {
                A[x][q] = *reinterpret_cast<const V*>(&L.A[q][row][kb]);
                B[x][q] = *reinterpret_cast<const V*>(&L.B[q][col][kb]);
            }
        }
#pragma unroll
        for (int y = 0; y < 2; ++y) {
            const V nbi = negate(B[y][1]);
            const V nbil = SPLIT ? negate(B[y][NP - 1]) : nbi;
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                // re: Ar Br - Ai Bi ; im: Ar Bi + Ai Br  (hi x hi)
                cr[x][y] = Mfma<T>::mac(A[x][0], B[y][0], cr[x][y]);
                cr[x][y] = Mfma<T>::mac(A[x][1], nbi, cr[x][y]);
                ci[x][y] = Mfma<T>::mac(A[x][0], B[y][1], ci[x][y]);
                ci[x][y] = Mfma<T>::mac(A[x][1], B[y][0], ci[x][y]);
                if constexpr (SPLIT) {
                    // hi x lo and lo x hi
                    cr[x][y] = Mfma<T>::mac(A[x][0], B[y][2], cr[x][y]);
                    cr[x][y] = Mfma<T>::mac(A[x][1], nbil, cr[x][y]);
                    cr[x][y] = Mfma<T>::mac(A[x][2], B[y][0], cr[x][y]);
                    cr[x][y] = Mfma<T>::mac(A[x][3], nbi, cr[x][y]);
                    ci[x][y] = Mfma<T>::mac(A[x][0], B[y][3], ci[x][y]);
                    ci[x][y] = Mfma<T>::mac(A[x][1], B[y][2], ci[x][y]);
                    ci[x][y] = Mfma<T>::mac(A[x][2], B[y][1], ci[x][y]);
                    ci[x][y] = Mfma<T>::mac(A[x][3], B[y][0], ci[x][y]);
                }
            }
        }
    }
}

// The factors of chunk c + 1 are generated into one LDS buffer while chunk c
// is contracted from the other: one barrier per chunk.  The points reach
// LDS two chunks ahead (double-buffered too) and are loaded into registers
// three chunks ahead.
template <typename T, bool SPLIT>
__global__ __launch_bounds__(MFMA_THREADS) void fresnel_mfma(MfmaArgs a) {
    typedef FrLds<T, SPLIT> Lds;
    constexpr int K = KCH<SPLIT>;
    extern __shared__ __attribute__((aligned(16))) unsigned char fr_dyn[];
    Lds* L = reinterpret_cast<Lds*>(fr_dyn);   // two buffers
    __shared__ double p_x[2][K], p_y[2][K], p_c[2][K];
    __shared__ float p_wr[2][K], p_wi[2][K];

    if (a.skip && *a.skip) return;
    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    const int wr = wave >> 1, wc = wave & 1;
    // XCD-aware order of the tiles: consecutive logical tiles on one XCD
    const int ntx = (a.nx + MC - 1) / MC;
    const int g = xcd_remap(blockIdx.x, gridDim.x);
    const int i0 = (g / ntx) * MR, j0 = (g % ntx) * MC;
    const bool full = i0 + MR <= a.ny && j0 + MC <= a.nx;
    const int64_t nch = a.npad / K;

    f32x16 cr[2][2], ci[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) {
            cr[x][y] = (f32x16)0.f;
            ci[x][y] = (f32x16)0.f;
        }
    auto stage_points = [&](int slot, const FrPoint& q) {
        p_x[slot][tid] = q.x;
        p_y[slot][tid] = q.y;
        p_c[slot][tid] = q.c;
        p_wr[slot][tid] = q.wre;
        p_wi[slot][tid] = q.wim;
    };
    auto generate = [&](int64_t c) {
        const int slot = (int)(c & 1);
        if (full)
            fr_generate_pairs<T, SPLIT, true, false>(L[slot], p_x[slot], p_y[slot], p_c[slot], p_wr[slot], p_wi[slot],
                                                     tid, i0, j0, a);
        else
            fr_generate_pairs<T, SPLIT, false, false>(L[slot], p_x[slot], p_y[slot], p_c[slot], p_wr[slot],
                                                      p_wi[slot], tid, i0, j0, a);
    };
    FrPoint nq{};
    if (tid < K) {
        if (nch > 0) stage_points(0, a.pts[tid]);
        if (nch > 1) stage_points(1, a.pts[K + tid]);
        if (nch > 2) nq = a.pts[2 * K + tid];
    }
    __syncthreads();
    if (nch > 0) generate(0);
    __syncthreads();
    for (int64_t c = 0; c < nch; ++c) {
        if (c + 1 < nch) generate(c + 1);
        fr_contract<T, SPLIT>(L[c & 1], wr, wc, lane, cr, ci);
        // slot c & 1 held chunk c's points, read by generate(c) one step ago
        if (tid < K && c + 2 < nch) {
            stage_points((int)(c & 1), nq);
            if (c + 3 < nch) nq = a.pts[(c + 3) * K + tid];
        }
        __syncthreads();
    }
    // epilogue
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int row = i0 + wr * 64 + 32 * x + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                const int col = j0 + wc * 64 + 32 * y + (lane & 31);
                if (row < a.ny && col < a.nx) a.out[(size_t)row * a.nx + col] = make_float2(cr[x][y][v], ci[x][y][v]);
            }
}

template <typename T, bool SPLIT>
int launch_fresnel_mfma(oph_ctx* ctx, const MfmaArgs& m, unsigned tiles) {
    const size_t shm = 2 * sizeof(FrLds<T, SPLIT>);
    static const bool attr = [&] {
        hipFuncSetAttribute(reinterpret_cast<const void*>(&fresnel_mfma<T, SPLIT>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
        hipGetLastError();
        return true;
    }();
    (void)attr;
    OPH_LAUNCH(ctx, "fresnel_mfma", (fresnel_mfma<T, SPLIT>), dim3(tiles), dim3(MFMA_THREADS), shm, m);
    return OPH_OK;
}

// ---------------------------------------------------------------------------
// Plane-factored contraction.  Points on one plane z_p share
// c_p = 1/(2 lambda z_p), and
//   A[i][n] = D_p(Y_i) w_n exp(i 2 pi c_p (y_n^2 - 2 Y_i y_n)),  D_p(Y) = exp(i 2 pi c_p Y^2),
// B likewise with X_j and x_n (no weight).  D_p is common to the plane's
// points, so the plane's part of the field is
//   U_p[i][j] = D_p(Y_i) D_p(X_j) sum_{n on p} g_n[i] h_n[j],
// and g, h are geometric along a run of rows (ratio exp(-i 2 pi 2 c_p y_n G p)):
// one complex multiply per entry instead of two.  The points are grouped by
// plane (a stable sort by z, so a plane's points keep their input order; each
// plane padded to whole 32-point chunks with zero-weight points), the
// contraction runs plane by plane, and at each plane's last chunk the
// accumulators are multiplied by D_p(Y_i) D_p(X_j) and added to the output.
// Partial sums per plane also keep the FP32 accumulation error of a long
// sum to the plane's share.  Used when the points lie on at most PLANE_MAX
// distinct planes with at least PLANE_MIN_AVG points per plane on average
// (the device decides after grouping, and the general kernel runs otherwise).
constexpr int PLANE_MAX = 4096;
constexpr int PLANE_MIN_AVG = 256;
constexpr int64_t PLANE_D_MAX = (int64_t)1 << 25;   // entries of the plane-chirp tables

__global__ void fr_keys(const double* z, int64_t n, unsigned long long* key, unsigned* idx) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    key[i] = (unsigned long long)__double_as_longlong(z[i]);
    idx[i] = (unsigned)i;
}

__global__ void fr_flags(const unsigned long long* key, int64_t n, unsigned* flag) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    flag[i] = (i == 0 || key[i] != key[i - 1]) ? 1u : 0u;
}

// pid[i] = 1 + plane of sorted point i; start of each plane, its c, the count
__global__ void fr_starts(const unsigned long long* key, const unsigned* flag, const unsigned* pid, int64_t n,
                          double lambda, unsigned* start, double* pc, int* info) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (flag[i]) {
        const unsigned p = pid[i] - 1;
        if (p < (unsigned)PLANE_MAX) {
            start[p] = (unsigned)i;
            pc[p] = 1.0 / (2.0 * lambda * __longlong_as_double((long long)key[i]));
        }
    }
    if (i == n - 1) info[1] = (int)min(pid[i], (unsigned)PLANE_MAX + 1);
}

// One workgroup: decides the form (info[0]) and pads each plane to whole
// chunks (poff: exclusive prefix of the padded counts).
__global__ __launch_bounds__(1024) void fr_plan(int64_t n, const unsigned* start, unsigned* poff, int* info,
                                                int64_t cap_chunks, int64_t dlen) {
    __shared__ unsigned part[1024];
    const int np = info[1];
    const int t = threadIdx.x;
    if (!(np >= 1 && np <= PLANE_MAX && (int64_t)np * PLANE_MIN_AVG <= n && (int64_t)np * dlen <= PLANE_D_MAX)) {
        if (t == 0) info[0] = 0;
        return;
    }
    unsigned pad[4], sum = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int q = 4 * t + j;
        const unsigned cnt = q < np ? (q + 1 < np ? start[q + 1] : (unsigned)n) - start[q] : 0u;
        pad[j] = (cnt + KC - 1) / KC * KC;
        sum += pad[j];
    }
    part[t] = sum;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const unsigned v = t >= off ? part[t - off] : 0u;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    const unsigned total = part[1023];
    if ((int64_t)(total / KC) > cap_chunks) {
        if (t == 0) info[0] = 0;
        return;
    }
    unsigned run = part[t] - sum;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int q = 4 * t + j;
        if (q < np) poff[q] = run;
        run += pad[j];
    }
    if (t == 0) {
        poff[np] = total;
        info[2] = (int)(total / KC);
        info[0] = 1;
    }
}

// grouped points: sorted point i to poff[p] + (i - start[p]); the tail of
// each plane's last chunk gets zero-weight points
__global__ void fr_fill(const double* x, const double* y, const double* z, const double* amp, const double* phase,
                        int64_t n, double lambda, const unsigned* order, const unsigned* pid, const unsigned* start,
                        const unsigned* poff, const double* pc, const int* info, FrPoint* pts) {
    if (!info[0]) return;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int np = info[1];
    if (i < n) {
        const unsigned p = pid[i] - 1;
        pts[poff[p] + (unsigned)(i - start[p])] = make_frpoint(x, y, z, amp, phase, order[i], lambda);
    }
    if (i < (int64_t)np * KC) {
        const int p = (int)(i / KC), r = (int)(i % KC);
        const unsigned cnt = (p + 1 < np ? start[p + 1] : (unsigned)n) - start[p];
        if (poff[p] + cnt + r < poff[p + 1]) pts[poff[p] + cnt + r] = zero_frpoint(pc[p]);
    }
}

// plane chirps D_p(Y_i) = exp(i 2 pi c_p Y_i^2) for the rows (dr[p ny + i])
// and D_p(X_j) for the columns (dc[p nx + j]), phases reduced in FP64
__global__ void fr_chirps(const double* pc, const int* info, int nx, int ny, double pitch, float2* dr, float2* dc) {
    if (!info[0]) return;
    const int np = info[1];
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nr = (int64_t)np * ny, ncl = (int64_t)np * nx;
    if (i >= nr + ncl) return;
    const bool row = i < nr;
    const int64_t e = row ? i : i - nr;
    const int len = row ? ny : nx;
    const int p = (int)(e / len), k = (int)(e % len);
    const double X = (k - len / 2) * pitch;
    double t = pc[p] * X * X;
    t -= rint(t);
    const float2 v = make_float2(cos_turns((float)t), sin_turns((float)t));
    if (row)
        dr[e] = v;
    else
        dc[e] = v;
}

struct PlaneMfmaArgs {
    const FrPoint* pts;   // grouped by plane, padded
    const unsigned* poff; // padded offset of each plane's first point (np + 1)
    const double* pc;     // c of each plane
    const int* info;      // [0] this form on, [1] planes, [2] 32-point chunks
    const float2* dr;     // plane chirps of the rows, [p ny + i]
    const float2* dc;     // and of the columns, [p nx + j]
    int nx, ny;
    double p;
    float2* out;
};

// The end of a plane: out (+)= D(Y) D(X) acc over the wave's 64 x 64 sub-tile
// (stored on the tile's first plane, added on the others), then acc = 0.
__device__ __forceinline__ void fr_flush(f32x16 (&cr)[2][2], f32x16 (&ci)[2][2], int pl, int wr, int wc, int lane,
                                         int i0, int j0, const PlaneMfmaArgs& a) {
    const bool first = pl == 0;
    // the lane index through a zero the compiler cannot see through: the
    // flush's addresses are the same at every plane and, hoisted out of the
    // chunk loop, would hold ~70 registers across it
    int zero;
    asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
    lane += zero;
    float2 dc[2];
    int col[2];
#pragma unroll
    for (int y = 0; y < 2; ++y) {
        col[y] = j0 + wc * 64 + 32 * y + (lane & 31);
        dc[y] = col[y] < a.nx ? a.dc[(size_t)pl * a.nx + col[y]] : make_float2(0.f, 0.f);
    }
    // four rows at a time: their chirps and previous outputs are all
    // requested before any is used (addresses clamped into the image, so no
    // branch guards a load; stores outside the image are skipped)
    const int cc0 = min(col[0], a.nx - 1), cc1 = min(col[1], a.nx - 1);
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int vg = 0; vg < 4; ++vg) {
            float2 dr[4], pv[4][2];
            int row[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                row[q] = i0 + wr * 64 + 32 * x + 8 * vg + 4 * (lane >> 5) + q;
                const int rc = min(row[q], a.ny - 1);
                dr[q] = a.dr[(size_t)pl * a.ny + rc];
                // (loaded on the first plane too, then not used: no branch)
                pv[q][0] = a.out[(size_t)rc * a.nx + cc0];
                pv[q][1] = a.out[(size_t)rc * a.nx + cc1];
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                asm volatile("" : "+v"(dr[q].x), "+v"(dr[q].y), "+v"(pv[q][0].x), "+v"(pv[q][0].y), "+v"(pv[q][1].x),
                             "+v"(pv[q][1].y));
                if (first) pv[q][0] = pv[q][1] = make_float2(0.f, 0.f);
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int v = 4 * vg + q;
#pragma unroll
                for (int y = 0; y < 2; ++y) {
                    const float2 d = make_float2(dr[q].x * dc[y].x - dr[q].y * dc[y].y,
                                                 dr[q].x * dc[y].y + dr[q].y * dc[y].x);
                    const float re = cr[x][y][v], im = ci[x][y][v];
                    const float2 val =
                        make_float2(pv[q][y].x + (re * d.x - im * d.y), pv[q][y].y + (re * d.y + im * d.x));
                    if (row[q] < a.ny && col[y] < a.nx) a.out[(size_t)row[q] * a.nx + col[y]] = val;
                }
            }
        }
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) {
            cr[x][y] = (f32x16)0.f;
            ci[x][y] = (f32x16)0.f;
        }
}

template <typename T, bool SPLIT>
__global__ __launch_bounds__(MFMA_THREADS) void fresnel_mfma_planes(PlaneMfmaArgs a) {
    typedef FrLds<T, SPLIT> Lds;
    constexpr int K = KCH<SPLIT>;
    if (!a.info[0]) return;
    extern __shared__ __attribute__((aligned(16))) unsigned char fr_dyn[];
    Lds* L = reinterpret_cast<Lds*>(fr_dyn);   // two buffers
    __shared__ double p_x[2][K], p_y[2][K], p_c[2][K];
    __shared__ float p_wr[2][K], p_wi[2][K];

    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    const int wr = wave >> 1, wc = wave & 1;
    const int ntx = (a.nx + MC - 1) / MC;
    const int g = xcd_remap(blockIdx.x, gridDim.x);
    const int i0 = (g / ntx) * MR, j0 = (g % ntx) * MC;
    const bool full = i0 + MR <= a.ny && j0 + MC <= a.nx;
    const int64_t nch = (int64_t)a.info[2] * (KC / K);
    // the current plane and its last K-point chunk
    int pl = 0;
    int64_t pend = (int64_t)(a.poff[1] / K) - 1;

    f32x16 cr[2][2], ci[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) {
            cr[x][y] = (f32x16)0.f;
            ci[x][y] = (f32x16)0.f;
        }
    auto stage_points = [&](int slot, const FrPoint& q) {
        p_x[slot][tid] = q.x;
        p_y[slot][tid] = q.y;
        p_c[slot][tid] = q.c;
        p_wr[slot][tid] = q.wre;
        p_wi[slot][tid] = q.wim;
    };
    auto generate = [&](int64_t c) {
        const int slot = (int)(c & 1);
        if (full)
            fr_generate_pairs<T, SPLIT, true, true>(L[slot], p_x[slot], p_y[slot], p_c[slot], p_wr[slot], p_wi[slot],
                                              tid, i0, j0, a);
        else
            fr_generate_pairs<T, SPLIT, false, true>(L[slot], p_x[slot], p_y[slot], p_c[slot], p_wr[slot], p_wi[slot],
                                               tid, i0, j0, a);
    };
    FrPoint nq{};
    if (tid < K) {
        if (nch > 0) stage_points(0, a.pts[tid]);
        if (nch > 1) stage_points(1, a.pts[K + tid]);
        if (nch > 2) nq = a.pts[2 * K + tid];
    }
    __syncthreads();
    if (nch > 0) generate(0);
    __syncthreads();
    for (int64_t c = 0; c < nch; ++c) {
        if (c + 1 < nch) generate(c + 1);
        fr_contract<T, SPLIT>(L[c & 1], wr, wc, lane, cr, ci);
        // slot c & 1 held chunk c's points, read by generate(c) one step ago
        if (tid < K && c + 2 < nch) {
            stage_points((int)(c & 1), nq);
            if (c + 3 < nch) nq = a.pts[(c + 3) * K + tid];
        }
        // the plane ends with its last chunk: flush, then the next plane's end
        // (a load once per plane, not per chunk: in the vector memory count it
        // would wait for the point prefetch)
        if (c == pend) {
            fr_flush(cr, ci, pl, wr, wc, lane, i0, j0, a);
            ++pl;
            if (pl < a.info[1]) pend = (int64_t)(a.poff[pl + 1] / K) - 1;
        }
        __syncthreads();
    }
}

template <typename T, bool SPLIT>
int launch_fresnel_mfma_planes(oph_ctx* ctx, const PlaneMfmaArgs& m, unsigned tiles) {
    const size_t shm = 2 * sizeof(FrLds<T, SPLIT>);
    static const bool attr = [&] {
        hipFuncSetAttribute(reinterpret_cast<const void*>(&fresnel_mfma_planes<T, SPLIT>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
        hipGetLastError();
        return true;
    }();
    (void)attr;
    OPH_LAUNCH(ctx, "fresnel_mfma", (fresnel_mfma_planes<T, SPLIT>), dim3(tiles), dim3(MFMA_THREADS), shm, m);
    return OPH_OK;
}

// Groups the points by plane (device side) and runs the plane-factored
// contraction; *info_out receives the device flag word the general path
// checks (its [0] is nonzero when this form produced the field).
int fresnel_planes(oph_ctx* ctx, int method, int nx, int ny, double pitch, double lambda, const double* dx,
                   const double* dy, const double* dz, const double* da, const double* dp, int64_t n, float2* out,
                   unsigned tiles, const int** info_out) {
    const int64_t cap_chunks = (n + (int64_t)PLANE_MAX * (KC - 1)) / KC + 1;
    char* w0 = static_cast<char*>(oph_scratch(ctx, SLOT_WORK0, 32 * (size_t)n + 256));
    char* tb = static_cast<char*>(oph_scratch(ctx, SLOT_TABLE, 16 * (PLANE_MAX + 1) + 256));
    // plane chirp tables: at most PLANE_D_MAX entries (the form is off beyond)
    const int64_t dlen = (int64_t)nx + ny;
    const int64_t dent = std::min<int64_t>((n / PLANE_MIN_AVG) * dlen, PLANE_D_MAX);
    float2* dtab = static_cast<float2*>(oph_scratch(ctx, SLOT_TABLE2, sizeof(float2) * (size_t)std::max<int64_t>(dent, 1)));
    if (!dtab) return OPH_ENOMEM;
    FrPoint* gp = static_cast<FrPoint*>(oph_scratch(ctx, SLOT_WORK1, sizeof(FrPoint) * cap_chunks * KC));
    if (!w0 || !tb || !gp) return OPH_ENOMEM;
    auto* kin = reinterpret_cast<unsigned long long*>(w0);
    auto* kout = kin + n;
    auto* iin = reinterpret_cast<unsigned*>(kout + n);
    unsigned* iout = iin + n;
    unsigned* flag = iout + n;
    unsigned* pid = flag + n;
    auto* pc = reinterpret_cast<double*>(tb);
    auto* start = reinterpret_cast<unsigned*>(pc + PLANE_MAX);
    unsigned* poff = start + PLANE_MAX + 1;
    int* info = reinterpret_cast<int*>(poff + PLANE_MAX + 1);
    size_t sort_bytes = 0, scan_bytes = 0;
    if (rocprim::radix_sort_pairs(nullptr, sort_bytes, kin, kout, iin, iout, (size_t)n, 0, 64, ctx->stream) !=
            hipSuccess ||
        rocprim::inclusive_scan(nullptr, scan_bytes, flag, pid, (size_t)n, rocprim::plus<unsigned>(), ctx->stream) !=
            hipSuccess)
        return oph_fail(ctx, OPH_EDEVICE, "plane grouping: temporary storage query failed");
    size_t tmp_bytes = std::max(sort_bytes, scan_bytes);
    void* tmp = oph_scratch(ctx, SLOT_AUX1, tmp_bytes);
    if (!tmp) return OPH_ENOMEM;
    const unsigned gb = (unsigned)((n + 255) / 256);
    OPH_LAUNCH(ctx, "fresnel_group", fr_keys, dim3(gb), dim3(256), 0, dz, n, kin, iin);
    if (rocprim::radix_sort_pairs(tmp, sort_bytes, kin, kout, iin, iout, (size_t)n, 0, 64, ctx->stream) !=
        hipSuccess)
        return oph_fail(ctx, OPH_EDEVICE, "plane grouping: sort failed");
    OPH_LAUNCH(ctx, "fresnel_group", fr_flags, dim3(gb), dim3(256), 0, kout, n, flag);
    if (rocprim::inclusive_scan(tmp, scan_bytes, flag, pid, (size_t)n, rocprim::plus<unsigned>(), ctx->stream) !=
        hipSuccess)
        return oph_fail(ctx, OPH_EDEVICE, "plane grouping: scan failed");
    OPH_LAUNCH(ctx, "fresnel_group", fr_starts, dim3(gb), dim3(256), 0, kout, flag, pid, n, lambda, start, pc,
               info);
    OPH_LAUNCH(ctx, "fresnel_group", fr_plan, dim3(1), dim3(1024), 0, n, start, poff, info, cap_chunks, dlen);
    const int64_t fill_n = std::max<int64_t>(n, (int64_t)PLANE_MAX * KC);
    OPH_LAUNCH(ctx, "fresnel_group", fr_fill, dim3((unsigned)((fill_n + 255) / 256)), dim3(256), 0, dx, dy, dz, da,
               dp, n, lambda, iout, pid, start, poff, pc, info, gp);
    // rows' tables first, then the columns': np (ny + nx) <= dent entries
    float2* dr = dtab;
    float2* dcl = dtab + (size_t)(dent / dlen) * ny;
    OPH_LAUNCH(ctx, "fresnel_group", fr_chirps, dim3((unsigned)((dent + 255) / 256)), dim3(256), 0, pc, info, nx, ny,
               pitch, dr, dcl);
    PlaneMfmaArgs m{};
    m.pts = gp;
    m.dr = dr;
    m.dc = dcl;
    m.poff = poff;
    m.pc = pc;
    m.info = info;
    m.nx = nx;
    m.ny = ny;
    m.p = pitch;
    m.out = out;
    int rc;
    switch (method) {
        case OPH_FRESNEL_MFMA_BF16: rc = launch_fresnel_mfma_planes<__bf16, false>(ctx, m, tiles); break;
        case OPH_FRESNEL_MFMA_BF16_SPLIT: rc = launch_fresnel_mfma_planes<__bf16, true>(ctx, m, tiles); break;
        case OPH_FRESNEL_MFMA_FP16: rc = launch_fresnel_mfma_planes<_Float16, false>(ctx, m, tiles); break;
        default: rc = launch_fresnel_mfma_planes<_Float16, true>(ctx, m, tiles); break;
    }
    if (rc) return rc;
    *info_out = info;
    return OPH_OK;
}

}  // namespace

extern "C" int oph_pc_fresnel(oph_ctx* ctx, int nx, int ny, double pitch, double lambda, const oph_points* pts,
                              int method, oph_c64* out, int flags) {
    int rc = oph_enter(ctx);
    if (rc) return rc;
    if (!pts || !out) return oph_fail(ctx, OPH_EINVAL, "null argument");
    if (nx <= 0 || ny <= 0 || nx > 65536 || ny > 65536) return oph_fail(ctx, OPH_EINVAL, "bad hologram size");
    if (!(pitch > 0) || !(lambda > 0)) return oph_fail(ctx, OPH_EINVAL, "bad pitch or wavelength");
    if (method < OPH_FRESNEL_VALU || method > OPH_FRESNEL_MFMA_FP16_SPLIT)
        return oph_fail(ctx, OPH_EINVAL, "unknown method %d", method);
    if (pts->n < 0 || (pts->n > 0 && (!pts->x || !pts->y || !pts->z)))
        return oph_fail(ctx, OPH_EINVAL, "bad point arrays");
    if ((flags & OPH_ASYNC) && !(flags & OPH_DEVICE_PTR))
        return oph_fail(ctx, OPH_EINVAL, "OPH_ASYNC needs device pointers");
    const int64_t n = pts->n;
    const int64_t npad = ((n + KC - 1) / KC) * KC;
    const size_t pb = (size_t)(n > 0 ? n : 1) * sizeof(double);
    const int sf = n > 0 ? flags : (flags | OPH_DEVICE_PTR);
    if (!(flags & OPH_DEVICE_PTR) && !oph_scratch(ctx, SLOT_PTS, 5 * pb)) return OPH_ENOMEM;
    const double* dx = static_cast<const double*>(oph_stage_in(ctx, SLOT_PTS, pts->x, pb, sf, 0));
    const double* dy = static_cast<const double*>(oph_stage_in(ctx, SLOT_PTS, pts->y, pb, sf, pb));
    const double* dz = static_cast<const double*>(oph_stage_in(ctx, SLOT_PTS, pts->z, pb, sf, 2 * pb));
    const double* da = static_cast<const double*>(oph_stage_in(ctx, SLOT_PTS, pts->amp, pb, sf, 3 * pb));
    const double* dp = static_cast<const double*>(oph_stage_in(ctx, SLOT_PTS, pts->phase, pb, sf, 4 * pb));
    if (n > 0 && (!dx || !dy || !dz)) return OPH_ENOMEM;
    FrPoint* fp = static_cast<FrPoint*>(oph_scratch(ctx, SLOT_AUX0, sizeof(FrPoint) * (npad > 0 ? npad : 1)));
    if (!fp) return OPH_ENOMEM;
    const size_t npix = (size_t)nx * ny;
    float2* o = reinterpret_cast<float2*>(out);
    if (!(flags & OPH_DEVICE_PTR)) {
        o = static_cast<float2*>(oph_scratch(ctx, SLOT_OUT, npix * sizeof(float2)));
        if (!o) return OPH_ENOMEM;
    }
    const unsigned tiles = (unsigned)(((nx + MC - 1) / MC) * ((ny + MR - 1) / MR));
    // MFMA forms: the plane-factored contraction when the points lie on few
    // planes (decided on the device; OPH_FRESNEL_PLANES=0 disables it), the
    // general one otherwise -- both are launched, the one not chosen returns
    const int* skip = nullptr;
    const char* pe = getenv("OPH_FRESNEL_PLANES");
    if (method != OPH_FRESNEL_VALU && n >= PLANE_MIN_AVG && n < ((int64_t)1 << 31) && !(pe && pe[0] == '0')) {
        rc = fresnel_planes(ctx, method, nx, ny, pitch, lambda, dx, dy, dz, da, dp, n, o, tiles, &skip);
        if (rc) return rc;
    }
    if (npad > 0)
        OPH_LAUNCH(ctx, "fresnel_prep", fresnel_prep, dim3((unsigned)((npad + 255) / 256)), dim3(256), 0, dx, dy,
                   dz, da, dp, n, npad, lambda, fp, skip);
    if (method == OPH_FRESNEL_VALU) {
        const int gx = (nx + F32_C - 1) / F32_C, gy = (ny + F32_R - 1) / F32_R;
        // points split over grid.z so that the resident workgroups (two per
        // CU) are filled: the split with the fewest point chunks per slot,
        // at least 1024 points each (1280 x 720, 20,000 points: 120 tiles in
        // 17 parts fill 3.98 of 4 rounds, 1.35 ms against 1.43 in 4 parts,
        // 0.94 of a round; four-product form) and at most 256 MiB of partial fields
        const int64_t tiles_f = (int64_t)gx * gy, slots = 2LL * std::max(ctx->cu_count, 1);
        int64_t chunks = 1;
        double best = 1e300;
        for (int64_t k = 1; k <= std::min<int64_t>(32, std::max<int64_t>(1, n / 1024)); ++k) {
            if (k > 1 && (size_t)k * npix > ((size_t)1 << 25)) break;
            const double cost = (double)((tiles_f * k + slots - 1) / slots) / (double)k;
            if (cost < best * 0.98) {
                best = cost;
                chunks = k;
            }
        }
        F32Args v{};
        v.pts = fp;
        v.npad = npad;
        v.chunk = std::max<int64_t>(KC, (npad / KC + chunks - 1) / chunks * KC);
        chunks = std::max<int64_t>(1, (npad + v.chunk - 1) / v.chunk);
        v.nx = nx;
        v.ny = ny;
        v.p = pitch;
        v.out = chunks == 1 ? o : static_cast<float2*>(oph_scratch(ctx, SLOT_WORK0, chunks * npix * sizeof(float2)));
        if (!v.out) return OPH_ENOMEM;
        OPH_LAUNCH(ctx, "fresnel_valu", fresnel_f32, dim3(gx, gy, (unsigned)chunks), dim3(256), 0, v);
        if (chunks > 1)
            OPH_LAUNCH(ctx, "fresnel_sum_chunks", fresnel_sum_chunks, dim3((unsigned)((npix + 255) / 256)), dim3(256),
                       0, v.out, (int)chunks, (int64_t)npix, o);
    } else {
        MfmaArgs m{};
        m.pts = fp;
        m.npad = npad;
        m.nx = nx;
        m.ny = ny;
        m.p = pitch;
        m.out = o;
        m.skip = skip;
        switch (method) {
            case OPH_FRESNEL_MFMA_BF16: rc = launch_fresnel_mfma<__bf16, false>(ctx, m, tiles); break;
            case OPH_FRESNEL_MFMA_BF16_SPLIT: rc = launch_fresnel_mfma<__bf16, true>(ctx, m, tiles); break;
            case OPH_FRESNEL_MFMA_FP16: rc = launch_fresnel_mfma<_Float16, false>(ctx, m, tiles); break;
            default: rc = launch_fresnel_mfma<_Float16, true>(ctx, m, tiles); break;
        }
        if (rc) return rc;
    }
    if (!(flags & OPH_DEVICE_PTR))
        OPH_HIP_CHECK(ctx, hipMemcpyAsync(out, o, npix * sizeof(float2), hipMemcpyDeviceToHost, ctx->stream));
    return oph_finish(ctx, flags);
}
