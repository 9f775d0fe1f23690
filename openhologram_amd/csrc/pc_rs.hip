// pc_rs.hip -- exact-distance Rayleigh-Sommerfeld point-cloud field on gfx950.
//
// Replaces the KETI generator loop (K/ophgen_pointcloud/ophgen_pointcloud.cpp:
// 195-249) and its CUDA kernel (K/ophgen_pointcloud_gpu/ophgen_pointcloud_gpu.cpp:
// 391-415).  Same field, different machine mapping:
//   * a workgroup owns a 64x64 pixel tile and accumulates the complex field in
//     registers (the reference does one global read-modify-write per point
//     per pixel); tiles far enough from the points sum them as a separable
//     contraction on the FP32 matrix cores (below), the others directly:
//   * each thread owns a 4x4 pixel block, points are staged 256 at a time in
//     LDS and read by broadcast;
//   * the phase k r needs ~1e6 rad of range at 1e-6 rad resolution, beyond
//     FP32: per (point, thread) the distance r0 to the block centre is formed
//     in FP64 and reduced to a fraction of a turn in FP64; per pixel the
//     offset r - r0 is the second-order expansion
//         (r - r0)/lambda = c1 q - c2 q^2,  q = r^2 - r0^2,
//         c1 = 1/(2 r0 lambda), c2 = 1/(8 r0^3 lambda)
//     in FP32 (q is a sum of a per-column and a per-row term), and sin/cos
//     are the hardware v_sin_f32/v_cos_f32, which take turns;
//   * a (thread, point) pair whose block is too close to the point for that
//     expansion (third-order term above 2e-8 turns, or |c1 q| above 16 turns)
//     takes an exact FP64 path per pixel;
//   * large point sets and small grids split the points over grid.z chunks;
//     a finalize kernel sums the chunks in a fixed order (deterministic),
//     applies the per-pixel tilt term in FP64 and writes the output format.
// The same kernel, with the amplitude divided by r per pixel and CWO's pixel
// grid, is cwoPLS::Huygens (CWO/cwoPLS.cpp:316-368):
//   U[i][j] = sum_n a_n exp(i (k r + ph + phi_n)) / r,
//   X_j = (j - nx/2) p, Y_i = (i - ny/2) p, r = |(X_j - x_n, Y_i - y_n, z_n + z)|;
// there 1/r = (1/r0)(1 + q/r0^2)^(-1/2) ~ (1/r0)(1 - q/(2 r0^2)) per pixel
// (relative error 3/8 (q/r0^2)^2 < 1e-8 wherever the phase expansion holds).
#include <algorithm>
#include <cmath>

#include "oph_internal.h"

namespace {

constexpr int TPB_X = 16, TPB_Y = 16;     // threads per workgroup
constexpr int BX = 4, BY = 4;             // pixels per thread
constexpr int TILE_X = TPB_X * BX, TILE_Y = TPB_Y * BY;
constexpr int PBATCH = TPB_X * TPB_Y;     // points staged per batch
constexpr int RS_MINPTS = 256;            // points per grid.z chunk, at least

struct RsArgs {
    const double* x;
    const double* y;
    const double* z;
    const double* amp;
    const double* phase;
    int64_t n;
    int64_t chunk;          // points per grid.z chunk
    double sx, sy, sz, oz;  // scale, offset
    int nx, ny;
    double px, py;
    // pixel centre X(col) = col px + x_off, Y(row) = ydir row py + y_off
    double x_off, y_off, ydir;
    double ph0;             // global phase, turns
    double inv_lambda;
    float2* partial;        // [chunks][ny][nx]
};

struct RsStage {
    double x[PBATCH], y[PBATCH], zz[PBATCH], ph[PBATCH];
    float a[PBATCH];
};

// A sin and cos per pixel and point, for tiles too close to the points for
// the contraction below.
template <bool HUYGENS>
__device__ __forceinline__ void rs_tile_direct(const RsArgs& a, RsStage& S) {
    double *s_x = S.x, *s_y = S.y, *s_zz = S.zz, *s_ph = S.ph;
    float* s_a = S.a;
    const int tid = threadIdx.x;
    const int tx = tid % TPB_X, ty = tid / TPB_X;
    const int c0 = blockIdx.x * TILE_X + tx * BX;
    const int r0 = blockIdx.y * TILE_Y + ty * BY;
    // block centre (KETI: X = (col + 1/2) px - Lx/2, Y = Ly/2 - (row + 1/2) py)
    const double X0 = (c0 + 0.5 * (BX - 1)) * a.px + a.x_off;
    const double Y0 = a.ydir * (r0 + 0.5 * (BY - 1)) * a.py + a.y_off;
    float ex[BX], ey[BY];
#pragma unroll
    for (int c = 0; c < BX; ++c) ex[c] = (float)((c - 0.5 * (BX - 1)) * a.px);
#pragma unroll
    for (int r = 0; r < BY; ++r) ey[r] = (float)(a.ydir * (r - 0.5 * (BY - 1)) * a.py);
    // largest |offset| in the block (for the expansion bound)
    const double hmax = 0.5 * sqrt((double)(BX - 1) * (BX - 1) * a.px * a.px +
                                   (double)(BY - 1) * (BY - 1) * a.py * a.py);
    const float hmaxf = (float)hmax;

    float re[BY][BX], im[BY][BX];
#pragma unroll
    for (int r = 0; r < BY; ++r)
#pragma unroll
        for (int c = 0; c < BX; ++c) re[r][c] = im[r][c] = 0.f;

    const int64_t p_begin = (int64_t)blockIdx.z * a.chunk;
    int64_t p_end = p_begin + a.chunk;
    if (p_end > a.n) p_end = a.n;
    const float inv_l_f = (float)a.inv_lambda;

    for (int64_t base = p_begin; base < p_end; base += PBATCH) {
        __syncthreads();
        {
            const int64_t j = base + tid;
            double xs = 0.0, ys = 0.0, zz = 1.0, ph = 0.0;
            float am = 0.f;
            if (j < p_end) {
                xs = a.x[j] * a.sx;
                ys = a.y[j] * a.sy;
                const double zs = a.z[j] * a.sz + a.oz;
                zz = zs * zs;
                am = a.amp ? (float)a.amp[j] : 1.f;
                ph = (a.phase ? a.phase[j] * 0.15915494309189535 : 0.0) + a.ph0;  // rad -> turns
            }
            s_x[tid] = xs;
            s_y[tid] = ys;
            s_zz[tid] = zz;
            s_ph[tid] = ph;
            s_a[tid] = am;
        }
        __syncthreads();
        const int cnt = (int)((p_end - base) < PBATCH ? (p_end - base) : PBATCH);
        for (int j = 0; j < cnt; ++j) {
            const double dx0 = X0 - s_x[j];
            const double dy0 = Y0 - s_y[j];
            const double s0 = fma(dx0, dx0, fma(dy0, dy0, s_zz[j]));
            const double yr = rsqrt_f64(s0);            // 1/r0
            const double rr0 = s0 * yr;                   // r0
            const double t0 = fma(rr0, a.inv_lambda, s_ph[j]);
            const float f0 = (float)(t0 - rint(t0));
            const float am = s_a[j];
            const float dxf = (float)dx0, dyf = (float)dy0;
            const double c1d = 0.5 * a.inv_lambda * yr;
            const float c1 = (float)c1d;
            const float yrf = (float)yr;
            const float c2 = 0.25f * c1 * yrf * yrf;
            // expansion bound: u = q/r0^2 <= (2 h rho + h^2)/r0^2; the
            // third-order term r0 u^3/(16 lambda) and the first-order size
            // c1 q (FP32 resolution) decide the path
            // Huygens amplitude: am/r0 (1 - q/(2 r0^2)) per pixel
            const float amr = HUYGENS ? am * yrf : am;
            const float hq = HUYGENS ? -0.5f * yrf * yrf : 0.f;
            const float rhof = __builtin_sqrtf(fmaf(dxf, dxf, dyf * dyf));
            const float qmax = fmaf(2.f * hmaxf, rhof, hmaxf * hmaxf);
            const float u = qmax * yrf * yrf;
            const bool exact = ((float)rr0 * u * u * u * (0.0625f * inv_l_f) > 2e-8f) || (c1 * qmax > 16.f);
            if (!exact) {
                float A[BX], B[BY];
#pragma unroll
                for (int c = 0; c < BX; ++c) A[c] = fmaf(2.f * ex[c], dxf, ex[c] * ex[c]);
#pragma unroll
                for (int r = 0; r < BY; ++r) B[r] = fmaf(2.f * ey[r], dyf, ey[r] * ey[r]);
#pragma unroll
                for (int r = 0; r < BY; ++r)
#pragma unroll
                    for (int c = 0; c < BX; ++c) {
                        const float q = A[c] + B[r];
                        const float ph = fmaf(q, fmaf(-c2, q, c1), f0);
                        const float ap = HUYGENS ? amr * fmaf(hq, q, 1.f) : am;
                        re[r][c] = fmaf(ap, cos_turns(ph), re[r][c]);
                        im[r][c] = fmaf(ap, sin_turns(ph), im[r][c]);
                    }
            } else {
#pragma unroll
                for (int r = 0; r < BY; ++r)
#pragma unroll
                    for (int c = 0; c < BX; ++c) {
                        const double dx = dx0 + (c - 0.5 * (BX - 1)) * a.px;
                        const double dy = dy0 + a.ydir * (r - 0.5 * (BY - 1)) * a.py;
                        const double s = fma(dx, dx, fma(dy, dy, s_zz[j]));
                        const double ys = rsqrt_f64(s);
                        const double t = fma(s * ys, a.inv_lambda, s_ph[j]);
                        const float ph = (float)(t - rint(t));
                        const float ap = HUYGENS ? (float)(am * ys) : am;
                        re[r][c] = fmaf(ap, cos_turns(ph), re[r][c]);
                        im[r][c] = fmaf(ap, sin_turns(ph), im[r][c]);
                    }
            }
        }
    }
    float2* dst = a.partial + (size_t)blockIdx.z * a.nx * a.ny;
#pragma unroll
    for (int r = 0; r < BY; ++r) {
        const int row = r0 + r;
        if (row >= a.ny) continue;
#pragma unroll
        for (int c = 0; c < BX; ++c) {
            const int col = c0 + c;
            if (col < a.nx) dst[(size_t)row * a.nx + col] = make_float2(re[r][c], im[r][c]);
        }
    }
}

// ---- separable contraction ------------------------------------------------
// Over a 32 x 32 pixel block the phase about the block centre is, with
// A = ex (2 dx + ex), B = ey (2 dy + ey) and q = A + B,
//   (r - r0)/lambda = c1 q - c2 q^2 + c3 q^3 - ...,
// c1 = 1/(2 r0 lambda), c2 = c1/(4 r0^2), c3 = c2/(2 r0^2): a part in A, a
// part in B, and the cross term -2 c2 A' B' with A' = A (1 - eta A),
// eta = 3/(4 r0^2) (third order included).  So
//   exp(i 2 pi r/lambda) = F(row) E(col) sum_k (i delta A' B')^k / k!,  delta = -4 pi c2,
// and the sum over points is a complex contraction of K = (points x terms) on
// v_mfma_f32_32x32x2_f32: per point and block 32 row and 32 column factors
// (a sin and cos each) instead of 1,024, one to five terms by the size of
// the cross term (one below 6e-7 rad; two up to 1.5e-3 rad cover a 100 mm
// distance at 8 um for most points).  The factors' phases are polynomials of
// the pixel offset j = -15.5 .. 15.5, FP32 with the linear coefficient,
// reduced modulo 2 in FP64 (2 j is odd, so j 2 is a whole turn), split so
// that its high part times j is exact, and so is that plus the high part of
// the centre phase: one rounding for each factor's phase.
//
// A wave owns a block.  It takes 64 points at a time: each lane forms one
// point's record for the block in FP64, then the wave contracts them in
// pairs (lanes 0-31 the factors of the even point, 32-63 of the odd one).
// Points out of the expansion's range (rs_terms) take the FP64 phase per
// pixel; a tile with more than 1/8 such points, by the sample, runs
// rs_tile_direct.  512^2 with 2000 points at 100 mm, a share of them at 3 mm:
// none 92 us, 6% 115, 9% 127, 11% 189, 13% 231, half 307, all 400, where the
// direct form for every tile took 455 to 867.
//
// The complex product takes three real ones instead of four, which costs the
// sums a factor 1.4 in rounding; they are formed over RS_BATCH points at a
// time and added per batch, which more than makes up for it.  Error against
// FP64 in the 2-norm at 1000 points: 2.2e-7 at 0.1 m, 2.0e-7 beyond 0.3 m
// (batches of 64: 3.5e-7 and 3.1e-7); one sum per pixel of 1000 products 6.6e-7
// and 5.8e-7.  At 100 points 2.1e-7 and 1.9e-7 (per pixel 3.9e-7 and 2.0e-7),
// at one 1.4e-7 and 1.3e-7 (2.3e-7 and 0.9e-7: the two factors' rounding is
// what is left, beyond 0.3 m more than that of one phase per pixel).
// Bound by matrix and vector instructions in turn (they do not overlap on a
// SIMD here).  1024^2 with 1000 points at 100 mm: 174 us (162 in batches of
// 64); 4096 x 2160 with 1453 points at 0.462 um: 1.85 ms (1.72).  A sin and
// cos per pixel and point took 457 us and 4.40 ms.  Records in the order of
// their terms are worth 8% (a pair takes the larger count of its two).

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int RS_TERMS = 5, RS_BATCH = 16;

struct RsRec {
    float4 x, y;   // high and low linear, quadratic, cubic coefficient along x and y
    float4 c;      // phase at the block centre, amplitude, quartic coefficients
    float4 m;      // 2 dx, 2 dy, delta, eta
    float c_lo;    // the centre phase's low part (the high part is a multiple of 2^-20)
    float pad[3];
};

// Terms the contraction needs for one point and block (0: out of range).
// ax, ay: largest A and B over the block; hm: largest half extent.  The
// thresholds keep the first dropped term, (delta A' B')^k / k!, whose root mean
// square over the block's 32 x 32 offsets is d^k / k! (32/31)^(2 k) / (2 k + 1),
// and the dropped phase terms (fourth order in q, fifth in the offset) below
// 3e-7 rad.
__device__ __forceinline__ int rs_terms(float r0, float yr, float c2, float ax, float ay, float dm, float hm,
                                        float inv_l, bool huygens) {
    const float u = (ax + ay) * yr * yr;
    const float c3 = 0.5f * c2 * yr * yr;
    const float e4 = r0 * inv_l * (5.f / 128.f) * (u * u) * (u * u);
    const float e5 = 8.f * c3 * dm * (hm * hm) * (hm * hm) * hm;
    if (!(e4 + e5 <= 5e-8f) || (huygens && !(u <= 1.5e-3f))) return 0;
    const float d = 12.5663706f * c2 * ax * ay;
    return d <= 6e-7f ? 1 : d <= 1.5e-3f ? 2 : d <= 2.1e-2f ? 3 : d <= 8e-2f ? 4 : d <= 0.18f ? 5 : 0;
}

template <bool HUYGENS>
__device__ __forceinline__ void rs_block_mfma(const RsArgs& a, RsRec* rec, int c0, int r0) {
    const int lane = threadIdx.x & 63;
    const double spy = a.ydir * a.py;
    const double X0 = (c0 + 15.5) * a.px + a.x_off, Y0 = (r0 + 15.5) * spy + a.y_off;
    const float hx = (float)(15.5 * a.px), hy = (float)(15.5 * a.py), hm = fmaxf(hx, hy);
    const float inv_l = (float)a.inv_lambda;
    // this lane's row and column offset (the same index of the block on both axes)
    const float j = (float)(lane & 31) - 15.5f;
    const float ex = j * (float)a.px, ey = j * (float)spy;
    f32x16 re = (f32x16)0.f, im = (f32x16)0.f;
    const int64_t p_begin = (int64_t)blockIdx.z * a.chunk;
    const int64_t p_end = min(a.n, p_begin + a.chunk);
    for (int64_t base = p_begin; base < p_end; base += 64) {
        int terms = 0;
        int first[RS_TERMS + 2];   // first record with at least k terms
        {
            const int64_t n = base + lane;
            RsRec q = {};
            if (n < p_end) {
                const double dx = X0 - a.x[n] * a.sx, dy = Y0 - a.y[n] * a.sy;
                const double zs = a.z[n] * a.sz + a.oz;
                const double s0 = fma(dx, dx, fma(dy, dy, zs * zs));
                const double yr = rsqrt_f64(s0), rr = s0 * yr;
                const double t0 = fma(rr, a.inv_lambda, (a.phase ? a.phase[n] * 0.15915494309189535 : 0.0) + a.ph0);
                const double c1 = 0.5 * a.inv_lambda * yr;
                const float yrf = (float)yr, y2 = yrf * yrf, c1f = (float)c1;
                const float c2 = 0.25f * c1f * y2, c3 = 0.5f * c2 * y2;
                const float dxf = (float)dx, dyf = (float)dy, pxf = (float)a.px, pyf = (float)spy;
                float am = a.amp ? (float)a.amp[n] : 1.f;
                if (HUYGENS) am *= yrf;
                auto axis = [&](double d, double p, float df, float pf, float& quartic) {
                    double s = 2.0 * c1 * d * p;
                    s -= 2.0 * rint(0.5 * s);
                    const double hi = rint(s * 131072.0) * (1.0 / 131072.0);
                    const float d2 = df * df, p2 = pf * pf;
                    quartic = fmaf(12.f * c3, d2, -c2) * p2 * p2;
                    return make_float4((float)hi, (float)(s - hi), fmaf(-4.f * c2, d2, c1f) * p2,
                                       df * fmaf(8.f * c3, d2, -4.f * c2) * p2 * pf);
                };
                float qx, qy;
                q.x = axis(dx, a.px, dxf, pxf, qx);
                q.y = axis(dy, spy, dyf, pyf, qy);
                const double tf = t0 - rint(t0), th = rint(tf * 1048576.0) * (1.0 / 1048576.0);
                q.c = make_float4((float)th, am, qx, qy);
                q.c_lo = (float)(tf - th);
                q.m = make_float4(2.f * dxf, 2.f * dyf, -12.5663706f * c2, 0.75f * y2);
                terms = rs_terms((float)rr, yrf, c2, hx * fmaf(2.f, fabsf(dxf), hx), hy * fmaf(2.f, fabsf(dyf), hy),
                                 fmaxf(fabsf(dxf), fabsf(dyf)), hm, inv_l, HUYGENS);
                // (an amplitude so large that the sums' products may overflow
                // where the point's value does not, infinite or NaN: inf - inf
                // would be NaN where the point adds +-inf)
                if (!(fabsf(am) <= 1e30f)) terms = 0;
                if (terms == 0) q = {};   // summed per pixel below
            }
            // records in order of their number of terms, so that the two points
            // of a pair mostly need the same; those of none (out of range, past
            // the end) last, with amplitude 0
            int at = 0, below = 0;
#pragma unroll
            for (int k = 1; k <= RS_TERMS + 1; ++k) {
                const uint64_t m = __ballot(terms == k % (RS_TERMS + 1));
                if (terms == k % (RS_TERMS + 1)) at = below + __popcll(m & ((1ull << lane) - 1));
                below += __popcll(m);
                if (k <= RS_TERMS) first[k + 1] = below;
            }
            rec[at] = q;
        }
        // (one wave's LDS accesses complete in order: only the compiler must
        // not move them)
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const int cnt = first[RS_TERMS + 1];
        // a complex product from three real ones: sums of fr er, fi ei and
        // (fr + fi)(er + ei), over RS_BATCH points
        f32x16 s1 = (f32x16)0.f, s2 = (f32x16)0.f, s3 = (f32x16)0.f;
        auto add_batch = [&]() {
            re += s1 - s2;
            im += s3 - (s1 + s2);
            s1 = s2 = s3 = (f32x16)0.f;
        };
        for (int p = 0; p < cnt; p += 2) {
            if (p > 0 && p % RS_BATCH == 0) add_batch();
            const RsRec q = rec[p + (lane >> 5)];
            float mx = j * q.x.x, my = fmaf(j, q.y.x, q.c.x);   // exact, both
            mx -= rintf(mx);
            my -= rintf(my);
            const float tx = fmaf(fmaf(fmaf(fmaf(q.c.z, j, q.x.w), j, q.x.z), j, q.x.y), j, mx);
            const float ty = fmaf(fmaf(fmaf(fmaf(q.c.w, j, q.y.w), j, q.y.z), j, q.y.y), j, q.c_lo) + my;
            float er = cos_turns(tx), ei = sin_turns(tx);
            float fr = q.c.y * cos_turns(ty), fi = q.c.y * sin_turns(ty);
            if (HUYGENS) {
                // 1/r = (1/r0)(1 - q/(2 r0^2) + 3/8 (q/r0^2)^2), per axis
                const float ua = ex * (q.m.x + ex) * q.m.w, ub = ey * (q.m.y + ey) * q.m.w;   // 3/4 A/r0^2
                const float ga = fmaf(ua, fmaf(ua, 2.f / 3.f, -2.f / 3.f), 1.f);
                const float gb = fmaf(ub, fmaf(ub, 2.f / 3.f, -2.f / 3.f), 1.f);
                er *= ga;
                ei *= ga;
                fr *= gb;
                fi *= gb;
            }
            auto contract = [&]() {
                s1 = __builtin_amdgcn_mfma_f32_32x32x2f32(fr, er, s1, 0, 0, 0);
                s2 = __builtin_amdgcn_mfma_f32_32x32x2f32(fi, ei, s2, 0, 0, 0);
                s3 = __builtin_amdgcn_mfma_f32_32x32x2f32(fr + fi, er + ei, s3, 0, 0, 0);
            };
            contract();
            if (p + 1 >= first[2]) {
                const float A = ex * (q.m.x + ex), B = ey * (q.m.y + ey);
                const float g = q.m.z * A * fmaf(-q.m.w, A, 1.f), b = B * fmaf(-q.m.w, B, 1.f);
                auto next = [&](float w) {   // E *= i g w, F *= b
                    const float gw = g * w, t = er;
                    er = -ei * gw;
                    ei = t * gw;
                    fr *= b;
                    fi *= b;
                    contract();
                };
                next(1.f);
                if (p + 1 >= first[3]) {
                    next(0.5f);
                    if (p + 1 >= first[4]) {
                        next(1.f / 3.f);
                        if (p + 1 >= first[5]) next(0.25f);
                    }
                }
            }
        }
        add_batch();
        // points out of range: FP64 phase per pixel (register v of a lane is
        // row 8 (v/4) + 4 (lane/32) + v%4, column lane%32)
        uint64_t far = __ballot(terms == 0 && base + lane < p_end);
        while (far) {
            const int k = __ffsll((long long)far) - 1;
            far &= far - 1;
            const int64_t n = base + k;
            const double dx = (c0 + (lane & 31)) * a.px + a.x_off - a.x[n] * a.sx;
            const double zs = a.z[n] * a.sz + a.oz, ys = a.y[n] * a.sy;
            const double dxz = fma(dx, dx, zs * zs);
            const double ph = (a.phase ? a.phase[n] * 0.15915494309189535 : 0.0) + a.ph0;
            const float am = a.amp ? (float)a.amp[n] : 1.f;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int row = r0 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                const double dy = row * spy + a.y_off - ys;
                const double s = fma(dy, dy, dxz), yr = rsqrt_f64(s);
                const double t = fma(s * yr, a.inv_lambda, ph);
                const float f = (float)(t - rint(t));
                const float ap = HUYGENS ? (float)(am * yr) : am;
                re[v] = fmaf(ap, cos_turns(f), re[v]);
                im[v] = fmaf(ap, sin_turns(f), im[v]);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    float2* dst = a.partial + (size_t)blockIdx.z * a.nx * a.ny;
    const int col = c0 + (lane & 31);
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const int row = r0 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
        if (row < a.ny && col < a.nx) dst[(size_t)row * a.nx + col] = make_float2(re[v], im[v]);
    }
}

// A 64 x 64 tile and one chunk of the points.  The form is chosen per
// workgroup from a sample of up to 256 of its points, spread over the chunk.
template <bool HUYGENS>
__global__ __launch_bounds__(256, 3) void rs_accumulate(RsArgs a) {
    __shared__ union {
        RsStage stage;
        RsRec rec[4][64];
    } sm;
    const int tile_x = blockIdx.x * TILE_X, tile_y = blockIdx.y * TILE_Y;
    const int64_t p_begin = (int64_t)blockIdx.z * a.chunk;
    const int64_t cnt = min(a.n, p_begin + a.chunk) - p_begin;
    bool out = false;
    const int64_t samples = min((int64_t)256, cnt);
    if ((int)threadIdx.x < samples) {
        const int64_t n = p_begin + cnt * threadIdx.x / samples;
        const float dx = (float)((tile_x + 31.5) * a.px + a.x_off - a.x[n] * a.sx);
        const float dy = (float)(a.ydir * (tile_y + 31.5) * a.py + a.y_off - a.y[n] * a.sy);
        const float zs = (float)(a.z[n] * a.sz + a.oz);
        const float s0 = fmaf(dx, dx, fmaf(dy, dy, zs * zs)), yr = rsqrtf(s0);
        const float hx = (float)(15.5 * a.px), hy = (float)(15.5 * a.py), inv_l = (float)a.inv_lambda;
        out = rs_terms(s0 * yr, yr, 0.125f * inv_l * yr * yr * yr, hx * fmaf(2.f, fabsf(dx), hx),
                       hy * fmaf(2.f, fabsf(dy), hy), fmaxf(fabsf(dx), fabsf(dy)), fmaxf(hx, hy), inv_l, HUYGENS) == 0;
    }
    const int n_out = __syncthreads_count(out);
    if (8 * (int64_t)n_out > samples) {
        rs_tile_direct<HUYGENS>(a, sm.stage);
        return;
    }
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c0 = tile_x + 32 * (wave & 1), r0 = tile_y + 32 * (wave >> 1);
    if (c0 < a.nx && r0 < a.ny) rs_block_mfma<HUYGENS>(a, sm.rec[wave], c0, r0);
}

struct FinArgs {
    const float2* partial;
    int chunks;
    int nx, ny;
    double px, py, half_lx, half_ly;
    double stx, sty, inv_lambda;  // sin(tilt)
    int tilt;
    void* out;
    int fmt;
    int accumulate;
};

// Sums the chunk partials in chunk order, applies exp(-i k (X sin tx + Y sin ty))
// and writes complex128 / complex64 / float Re.
__global__ __launch_bounds__(256) void rs_finalize(FinArgs f) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t npix = (int64_t)f.nx * f.ny;
    if (i >= npix) return;
    double re = 0.0, im = 0.0;
    for (int c = 0; c < f.chunks; ++c) {
        const float2 v = f.partial[(size_t)c * npix + i];
        re += v.x;
        im += v.y;
    }
    if (f.tilt) {
        const int row = (int)(i / f.nx), col = (int)(i % f.nx);
        const double X = (col + 0.5) * f.px - f.half_lx;
        const double Y = f.half_ly - (row + 0.5) * f.py;
        const double t = (X * f.stx + Y * f.sty) * f.inv_lambda;
        const float ft = (float)(t - rint(t));
        const double cs = cos_turns(ft), sn = -(double)sin_turns(ft);
        const double nr = re * cs - im * sn, ni = re * sn + im * cs;
        re = nr;
        im = ni;
    }
    if (f.fmt == OPH_OUT_C128) {
        double2* o = static_cast<double2*>(f.out) + i;
        if (f.accumulate) { double2 p = *o; re += p.x; im += p.y; }
        *o = make_double2(re, im);
    } else if (f.fmt == OPH_OUT_C64) {
        float2* o = static_cast<float2*>(f.out) + i;
        if (f.accumulate) { float2 p = *o; re += p.x; im += p.y; }
        *o = make_float2((float)re, (float)im);
    } else {
        float* o = static_cast<float*>(f.out) + i;
        float v = (float)re;
        if (f.accumulate) v += *o;
        *o = v;
    }
}

}  // namespace

namespace {

// Shared host side of oph_pc_rs and oph_pc_huygens: argument checks, point
// staging, the accumulate launch (KETI or CWO pixel grid, with or without
// 1/r) and the finalize launch.
struct RsJob {
    int nx, ny;
    double px, py, lambda;
    double scale[3], offset_z;
    double tilt_deg[2];
    bool cwo_grid, huygens;
    double ph0;  // global phase (radians)
};

int rs_run(oph_ctx* ctx, const RsJob& J, const oph_points* pts, void* out, int flags) {
    if (!pts || !out) return oph_fail(ctx, OPH_EINVAL, "null argument");
    if (J.nx <= 0 || J.ny <= 0 || J.nx > 65536 || J.ny > 65536)
        return oph_fail(ctx, OPH_EINVAL, "image size %dx%d out of range", J.nx, J.ny);
    if (!(J.px > 0) || !(J.py > 0) || !(J.lambda > 0))
        return oph_fail(ctx, OPH_EINVAL, "pitch and wavelength must be positive");
    if (pts->n < 0 || (pts->n > 0 && (!pts->x || !pts->y || !pts->z)))
        return oph_fail(ctx, OPH_EINVAL, "bad point arrays");
    const int fmt = flags & OPH_OUT_MASK;
    if (fmt != OPH_OUT_C128 && fmt != OPH_OUT_C64 && fmt != OPH_OUT_FRINGE)
        return oph_fail(ctx, OPH_EINVAL, "bad output format flag");
    if ((flags & OPH_ASYNC) && !(flags & OPH_DEVICE_PTR))
        return oph_fail(ctx, OPH_EINVAL, "OPH_ASYNC needs device pointers");

    const int nx = J.nx, ny = J.ny;
    const int64_t n = pts->n;
    const size_t npix = (size_t)nx * ny;
    const size_t pbytes = (size_t)(n > 0 ? n : 1) * sizeof(double);

    RsArgs a{};
    a.n = n;
    if (!(flags & OPH_DEVICE_PTR) && !oph_scratch(ctx, SLOT_PTS, 5 * pbytes)) return OPH_ENOMEM;
    const int sflags = n > 0 ? flags : (flags | OPH_DEVICE_PTR);  // nothing to copy when n == 0
    a.x = static_cast<const double*>(oph_stage_in(ctx, SLOT_PTS, pts->x, pbytes, sflags, 0 * pbytes));
    a.y = static_cast<const double*>(oph_stage_in(ctx, SLOT_PTS, pts->y, pbytes, sflags, 1 * pbytes));
    a.z = static_cast<const double*>(oph_stage_in(ctx, SLOT_PTS, pts->z, pbytes, sflags, 2 * pbytes));
    a.amp = static_cast<const double*>(oph_stage_in(ctx, SLOT_PTS, pts->amp, pbytes, sflags, 3 * pbytes));
    a.phase = static_cast<const double*>(oph_stage_in(ctx, SLOT_PTS, pts->phase, pbytes, sflags, 4 * pbytes));
    if (n > 0 && (!a.x || !a.y || !a.z)) return OPH_ENOMEM;
    if (n > 0 && ((pts->amp && !a.amp) || (pts->phase && !a.phase))) return OPH_ENOMEM;

    a.sx = J.scale[0];
    a.sy = J.scale[1];
    a.sz = J.scale[2];
    a.oz = J.offset_z;
    a.nx = nx;
    a.ny = ny;
    a.px = J.px;
    a.py = J.py;
    const double half_lx = J.px * nx / 2.0, half_ly = J.py * ny / 2.0;
    if (J.cwo_grid) {
        // cwoPLS: X = (col - nx/2) p, Y = (row - ny/2) p (CWO/cwoPLS.cpp:350-351)
        a.x_off = -(double)(nx / 2) * J.px;
        a.y_off = -(double)(ny / 2) * J.py;
        a.ydir = 1.0;
    } else {
        // KETI: X = (col + 1/2) p - Lx/2, Y = Ly/2 - (row + 1/2) p
        a.x_off = 0.5 * J.px - half_lx;
        a.y_off = half_ly - 0.5 * J.py;
        a.ydir = -1.0;
    }
    a.ph0 = J.ph0 * 0.15915494309189535;
    a.inv_lambda = 1.0 / J.lambda;

    const int gx = (nx + TILE_X - 1) / TILE_X, gy = (ny + TILE_Y - 1) / TILE_Y;
    const int64_t tiles = (int64_t)gx * gy;
    // split points so that the grid holds >= 4 workgroups per CU, keeping
    // >= RS_MINPTS points per chunk (1024^2, 1000 points: 4 chunks of 250;
    // 128 or 256 points at least and 2, 4 or 8 workgroups per CU measured the
    // same to 2%)
    int64_t chunks = (4LL * ctx->cu_count + tiles - 1) / tiles;
    const int64_t max_by_pts = (n + RS_MINPTS - 1) / RS_MINPTS;
    if (chunks > max_by_pts) chunks = max_by_pts;
    if (chunks > 16) chunks = 16;
    if (chunks < 1) chunks = 1;
    a.chunk = (n + chunks - 1) / chunks;
    if (a.chunk < 1) a.chunk = 1;
    a.partial = static_cast<float2*>(oph_scratch(ctx, SLOT_WORK0, chunks * npix * sizeof(float2)));
    if (!a.partial) return OPH_ENOMEM;

    if (J.huygens)
        OPH_LAUNCH(ctx, "huygens_accumulate", rs_accumulate<true>, dim3(gx, gy, (unsigned)chunks),
                   dim3(256), 0, a);
    else
        OPH_LAUNCH(ctx, "rs_accumulate", rs_accumulate<false>, dim3(gx, gy, (unsigned)chunks),
                   dim3(256), 0, a);

    const size_t obytes = npix * (fmt == OPH_OUT_C128 ? 16 : fmt == OPH_OUT_C64 ? 8 : 4);
    void* dout = out;
    if (!(flags & OPH_DEVICE_PTR)) {
        dout = oph_scratch(ctx, SLOT_OUT, obytes);
        if (!dout) return OPH_ENOMEM;
        if (flags & OPH_ACCUMULATE)
            OPH_HIP_CHECK(ctx, hipMemcpyAsync(dout, out, obytes, hipMemcpyHostToDevice, ctx->stream));
    }
    FinArgs f{};
    f.partial = a.partial;
    f.chunks = (int)chunks;
    f.nx = nx;
    f.ny = ny;
    f.px = a.px;
    f.py = a.py;
    f.half_lx = half_lx;
    f.half_ly = half_ly;
    f.stx = sin(J.tilt_deg[0] * (M_PI / 180.0));
    f.sty = sin(J.tilt_deg[1] * (M_PI / 180.0));
    f.inv_lambda = a.inv_lambda;
    f.tilt = (f.stx != 0.0 || f.sty != 0.0);
    f.out = dout;
    f.fmt = fmt;
    f.accumulate = (flags & OPH_ACCUMULATE) ? 1 : 0;
    OPH_LAUNCH(ctx, "rs_finalize", rs_finalize, dim3((unsigned)((npix + 255) / 256)), dim3(256), 0, f);
    if (!(flags & OPH_DEVICE_PTR))
        OPH_HIP_CHECK(ctx, hipMemcpyAsync(out, dout, obytes, hipMemcpyDeviceToHost, ctx->stream));
    return oph_finish(ctx, flags);
}

}  // namespace

extern "C" int oph_pc_rs(oph_ctx* ctx, const oph_spec* spec, const oph_points* pts, void* out,
                         int flags) {
    int rc = oph_enter(ctx);
    if (rc) return rc;
    if (!spec) return oph_fail(ctx, OPH_EINVAL, "null argument");
    RsJob J{};
    J.nx = spec->nx;
    J.ny = spec->ny;
    J.px = spec->pitch_x;
    J.py = spec->pitch_y;
    J.lambda = spec->lambda;
    for (int k = 0; k < 3; ++k) J.scale[k] = spec->scale[k];
    J.offset_z = spec->offset_z;
    J.tilt_deg[0] = spec->tilt_deg[0];
    J.tilt_deg[1] = spec->tilt_deg[1];
    return rs_run(ctx, J, pts, out, flags);
}

extern "C" int oph_pc_huygens(oph_ctx* ctx, int nx, int ny, double pitch, double lambda, double z, double ph,
                              const oph_points* pts, void* out, int flags) {
    int rc = oph_enter(ctx);
    if (rc) return rc;
    if ((flags & OPH_OUT_MASK) == OPH_OUT_FRINGE)
        return oph_fail(ctx, OPH_EINVAL, "oph_pc_huygens writes complex output only");
    RsJob J{};
    J.nx = nx;
    J.ny = ny;
    J.px = J.py = pitch;
    J.lambda = lambda;
    J.scale[0] = J.scale[1] = J.scale[2] = 1.0;
    J.offset_z = z;
    J.cwo_grid = true;
    J.huygens = true;
    J.ph0 = ph;
    return rs_run(ctx, J, pts, out, flags);
}
